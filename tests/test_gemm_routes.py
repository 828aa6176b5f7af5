"""Which kernel a product runs on, asked of the library on the host (tmb_gemm_route; the launches follow
the same choice)."""

import itertools

import pytest

SIMT, RING, TRANSPOSED_A, SPLITK, SMALL, ANY, STREAM64, F32, F32_WIDE = range(9)
PLENTY = 1 << 40   # more scratch than any plan asks for


def _ek():
    from torch_mojo_backend import eager_kernels as ek
    return ek


def route(m, n, k, ta=0, tb=0, dtype=None, batch=1, lda=None, ldb=None, a_aligned=1, b_aligned=1, epilogue=0,
          residual=0, workspace=0):
    """(kernel, tile, splits), or the negative status."""
    ek = _ek()
    lda = lda or (m if ta else k)
    ldb = ldb or (k if tb else n)
    r = ek.lib().tmb_gemm_route(batch, m, n, k, lda, ldb, m * k if batch > 1 else 0, k * n if batch > 1 else 0,
                                a_aligned, b_aligned, ta, tb, ek.BF16 if dtype is None else dtype, epilogue, residual,
                                workspace)
    return r if r < 0 else (r & 0xff, r >> 8 & 0xff, r >> 16)


def test_routes_of_known_products():
    ek = _ek()
    assert route(8192, 8192, 8192)[0] == RING
    assert route(128, 768, 768)[0] == SMALL
    assert route(8192, 3072, 16384, ta=1)[0] == TRANSPOSED_A
    assert route(768, 3072, 16384, ta=1, workspace=PLENTY)[0] == SPLITK
    assert route(768, 768, 32768, ta=1, workspace=PLENTY) == (SPLITK, 0, 14)       # 128 x 128 tiles
    assert route(3072, 768, 8192, ta=1, workspace=PLENTY) == (SPLITK, 1, 7)        # 256 x 256
    assert route(100, 77, 50, a_aligned=0)[0] == ANY
    assert route(8192, 4096, 64)[0] == STREAM64
    assert route(4, 4, 4, b_aligned=0)[0] == SIMT            # fewer than eight contiguous elements
    assert route(333, 77, 50, dtype=ek.F32)[0] == F32
    assert route(4096, 4096, 4096, dtype=ek.F32)[0] == F32_WIDE
    assert route(3, 3, 3, dtype=ek.F32)[0] == SIMT
    assert route(3, 3, 3, dtype=ek.F32, residual=1) == ek.ERR_UNSUPPORTED
    assert route(4, 4, 4, dtype=ek.I64) == ek.ERR_UNSUPPORTED
    assert route(4, 4, 0) == route(4, 0, 4) == route(4, 8, 8, lda=4) == ek.ERR_INVALID_ARGUMENT


def test_the_shapes_of_the_gpu_tests_take_every_tile():
    """One per tile of each kernel, in each layout: a refit of the models' constants must not drop one."""
    import test_hip_gemm
    import test_hip_gemm_any
    import test_hip_gemm_f32_edges
    import test_hip_gemm_small
    from torch_mojo_backend.eager_kernels import hip_ops
    ek = _ek()
    off = dict(a_aligned=0, b_aligned=0, workspace=PLENTY)
    for ta, tb in itertools.product((0, 1), repeat=2):
        took = [route(*mnk, ta=ta, tb=tb, **off) for mnk in test_hip_gemm_any.SHAPES]
        assert {t for kernel, t, _ in took if kernel == ANY} == set(range(5)) and max(t[2] for t in took) > 1
        took = [route(*mnk, ta=ta, tb=tb, dtype=ek.F32, **off) for mnk in test_hip_gemm_f32_edges.SHAPES]
        assert {t for kernel, t, _ in took if kernel == F32} == set(range(4)) and max(t[2] for t in took) > 1
        assert ta or {route(*mnk, tb=tb) for mnk in test_hip_gemm_small.SHAPES} == {(SMALL, t, 0) for t in range(6)}
    took = {(ta, tb, *route(m, n, k, int(ta), int(tb), workspace=PLENTY)[:2]) for m, n, k, ta, tb in test_hip_gemm.SPLITK}
    assert took == {(ta, tb, SPLITK, t) for ta, tb in ((False, False), (False, True), (True, False)) for t in (0, 1)}
    # which products of awkward layouts are copied first
    for dtype, a, ta, b, tb, padded in test_hip_gemm.AWKWARD:
        m, k = (a[-1], a[-2]) if ta else a[-2:]
        n, batch = (b[-2] if tb else b[-1]), (a[0] if len(a) == 3 else 1)
        form = (batch, m, n, k, m if ta else k, k if tb else n, 1, 1, int(ta), int(tb))
        if dtype.itemsize == 4:
            assert ek.lib().tmb_gemm_f32_padding_pays(*form) == padded, form
        else:
            assert (ek.lib().tmb_gemm_in_place_workspace_bytes(*form, 1, hip_ops.code_of(dtype)) < 0) == padded, form


@pytest.mark.parametrize("dtype_name", ["BF16", "F16", "F32"])
def test_the_scratch_a_caller_is_told_of_is_what_the_launch_splits_with(dtype_name):
    ek = _ek()
    dtype = getattr(ek, dtype_name)
    split = 0
    for m, n, k, ta, tb in itertools.product((1, 8, 100, 264, 768, 1024, 4096), (8, 72, 768, 3072), (64, 768, 3072, 16384),
                                             (0, 1), (0, 1)):
        told = ek.lib().tmb_gemm_layout_workspace_bytes(1, m, n, k, ta, tb, dtype)
        full, given, none = (route(m, n, k, ta, tb, dtype, workspace=w) for w in (PLENTY, told, 0))
        assert none[2] == 0
        if full[0] == ANY:
            continue    # a transposed A that the aligned kernels do not take: another entry sizes its scratch
        assert given == full, (m, n, k, ta, tb)
        assert full[2] * m * n * 4 in (0, told)
        split += full[2] > 0
    assert split > 20


@pytest.mark.parametrize("seed", range(4))
def test_scratch_for_an_unknown_layout_is_enough_for_every_layout(seed):
    """fp32, whose splits do not depend on the layout: what tmb_gemm_workspace_bytes answers splits as far as any
    amount does, and is no more than that."""
    import math
    import random
    ek, rng = _ek(), random.Random(seed)
    shapes = [(31, 67, 12565), (12, 1272, 1974), (245, 4220, 13614), (100, 72, 8200), (1024, 768, 3072), (2759, 3965, 26572)]
    shapes += [tuple(round(math.exp(rng.uniform(math.log(4), math.log(30000)))) for _ in range(3)) for _ in range(300)]
    split = 0
    for m, n, k in shapes:
        told = ek.lib().tmb_gemm_workspace_bytes(1, m, n, k, ek.F32)
        most = 0
        for ta, tb, aligned in itertools.product((0, 1), repeat=3):
            form = dict(ta=ta, tb=tb, dtype=ek.F32, a_aligned=aligned)
            full = route(m, n, k, workspace=PLENTY, **form)
            assert route(m, n, k, workspace=told, **form) == full, (m, n, k, form)
            most = max(most, full[2])
            by_layout = ek.lib().tmb_gemm_layout_workspace_bytes(1, m, n, k, ta, tb, ek.F32)
            if aligned or by_layout:
                assert route(m, n, k, workspace=by_layout, **form) == full, (m, n, k, form)
        assert told == most * m * n * 4, (m, n, k)
        split += most > 0
    assert split > 30


def test_a_large_transposed_a_with_a_residual_is_multiplied_and_added():
    """The rings take such a product without a residual only; the any-layout kernel, which takes it with
    one, is behind the two launches once the product is large."""
    ek = _ek()
    for residual_step in (0, ek.EPI_ROUND_LIKE_UNFUSED):
        large = dict(ta=1, residual=1, epilogue=residual_step, workspace=PLENTY)
        assert route(4096, 4096, 4096, **large) == ek.ERR_UNSUPPORTED
        assert route(50304, 768, 16384, **large) == ek.ERR_UNSUPPORTED
        assert route(768, 3072, 16384, **large)[0] == SPLITK         # its reduction adds the residual
        assert route(4097, 4096, 4096, **large)[0] == ANY            # the rings do not take it either way
    assert route(256, 256, 256, ta=1, residual=1)[0] == ANY          # one launch instead of the product and an add in float32
    assert route(768, 3072, 1024, ta=1, residual=1)[0] == ANY
    rounded = dict(ta=1, residual=1, epilogue=ek.EPI_ROUND_LIKE_UNFUSED)
    assert route(256, 256, 256, **rounded) == ek.ERR_UNSUPPORTED     # (the bits of the rings' product)


def test_a_transposed_a_with_a_gelu_does_not_fall_back_where_one_round_takes_the_product_alone():
    """The reduction of a split launch evaluates it, or, where it is to have the bits of two operations, the tiles that the
    product alone runs on; the any-layout kernel is 1.5 times as long."""
    ek = _ek()
    for m, n, k in ((3072, 768, 2048), (2304, 768, 2048), (2304, 1024, 3072), (3072, 768, 4096)):
        plain = dict(ta=1, workspace=PLENTY)
        for step in (0, ek.EPI_ROUND_LIKE_UNFUSED):
            assert route(m, n, k, epilogue=step, **plain)[0] == TRANSPOSED_A, (m, n, k)
        for gelu in (ek.EPI_GELU_TANH, ek.EPI_GELU_ERF):
            assert route(m, n, k, epilogue=gelu, **plain)[0] == SPLITK, (m, n, k)
            assert route(m, n, k, epilogue=gelu | ek.EPI_ROUND_LIKE_UNFUSED, **plain)[0] == TRANSPOSED_A, (m, n, k)
            assert route(m, n, k, epilogue=gelu | ek.EPI_ROUND_LIKE_UNFUSED, ta=1)[0] == ANY


ONE_ROUND = [(3072, 768, 2048), (3064, 776, 2304), (3072, 768, 4096)]    # (m, n, k) of a transposed A, else split


def test_a_residual_on_a_transposed_a_is_carried_where_a_split_launch_carried_it():
    ek = _ek()
    for m, n, k in ONE_ROUND:
        told = ek.lib().tmb_gemm_layout_workspace_bytes(1, m, n, k, 1, 0, ek.BF16)
        rounded = dict(ta=1, residual=1, epilogue=ek.EPI_ROUND_LIKE_UNFUSED)
        assert route(m, n, k, ta=1, workspace=told) == (TRANSPOSED_A, 0, 0)
        assert route(m, n, k, workspace=told, **rounded) == (TRANSPOSED_A, 0, 0)
        assert route(m, n, k, **rounded) == ek.ERR_UNSUPPORTED       # without the scratch, as ever
        assert route(m, n, k, ta=1, residual=1, workspace=told)[0] == SPLITK


@pytest.mark.gpu
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
@pytest.mark.parametrize("mnk", ONE_ROUND)
def test_that_residual_and_a_gelu_have_the_bits_of_two_operations(mnk, dtype_name):
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    m, n, k = mnk
    g = torch.Generator(device="cuda").manual_seed(k)
    x, w, bias, r = (torch.randn(*s, generator=g, device="cuda").to(getattr(torch, dtype_name))
                     for s in ((k, m), (k, n), (n,), (m, n)))
    out, ws = torch.empty_like(r), torch.empty(128 << 20, dtype=torch.uint8, device="cuda")
    ek = _ek()
    code = hip_ops.code_of(r.dtype)
    for b in (None, bias):
        assert ek.lib().tmb_gemm_residual_ws(
            out.data_ptr(), x.data_ptr(), w.data_ptr(), None if b is None else b.data_ptr(), r.data_ptr(), 1, m, n, k, m, n,
            n, n, 0, 0, 0, 0, 1, 0, code, code, code, ek.EPI_ROUND_LIKE_UNFUSED, ws.data_ptr(), ws.numel(),
            torch.cuda.current_stream().cuda_stream) == 0
        plain = hip_ops.gemm(x.t(), w, b)
        assert torch.equal(out, plain + r)
        for gelu, approximate in ((ek.EPI_GELU_TANH, "tanh"), (ek.EPI_GELU_ERF, "none")):
            assert ek.lib().tmb_gemm_ws(
                out.data_ptr(), x.data_ptr(), w.data_ptr(), None if b is None else b.data_ptr(), 1, m, n, k, m, n, n, 0, 0,
                0, 1, 0, code, gelu | ek.EPI_ROUND_LIKE_UNFUSED, ws.data_ptr(), ws.numel(),
                torch.cuda.current_stream().cuda_stream) == 0
            assert torch.equal(out, hip_ops.gelu(plain, approximate))


@pytest.mark.parametrize("dtype_name", ["BF16", "F16", "F32"])
def test_a_residual_that_is_added_with_the_bits_of_two_operations_is_carried_where_the_product_runs(dtype_name):
    """fp32, and 16-bit with TMB_EPI_ROUND_LIKE_UNFUSED: the kernel, tile and splits of the product alone, or none; all
    layouts, alignments, with and without scratch."""
    ek = _ek()
    dtype = getattr(ek, dtype_name)
    carried = apart = 0
    for batch, m, n, k in itertools.product((1, 5), (8, 100, 768, 4096), (16, 333, 2048), (8, 64, 100, 768, 4096)):
        for ta, tb, aa, ba, ws in itertools.product((0, 1), repeat=5):
            form = dict(ta=ta, tb=tb, a_aligned=aa, b_aligned=ba, workspace=ws * PLENTY, batch=batch, dtype=dtype)
            plain = route(m, n, k, **form)
            with_it = route(m, n, k, residual=1, epilogue=ek.EPI_ROUND_LIKE_UNFUSED, **form)
            if plain[0] == STREAM64:
                assert with_it[0] == RING      # (adds its four steps of K in the same order)
            elif with_it == ek.ERR_UNSUPPORTED:
                assert plain[0] in (SIMT, TRANSPOSED_A, F32_WIDE)
                apart += 1
            else:
                assert with_it == plain, (batch, m, n, k, form)
                carried += 1
    assert carried > 500 and apart > 100


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(256, 256, 256), (2048, 2048, 512), (4096, 2048, 2048)])
def test_transposed_a_with_a_residual_matches_float64(mnk):
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    m, n, k = mnk
    g = torch.Generator(device="cuda").manual_seed(m)
    x, w, bias, r = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((k, m), (k, n), (n,), (m, n)))
    plain = hip_ops.gemm(x.t(), w, bias)
    exact = x.double().t().contiguous() @ w.double() + bias.double()
    slack = (k + 2) * 2.0 ** -24 * (x.double().abs().t().contiguous() @ w.double().abs() + exact.abs()) + 1e-6
    step = hip_ops.gemm(x.t(), w, bias, residual=r, round_like_unfused=True)
    # rounded after the product (2^-9 of it) and after the sum
    exact_step = exact + r.double()
    assert ((step.double() - exact_step).abs() <= 2 * slack + 2.0 ** -8 * (exact.abs() + exact_step.abs())).all()
    assert torch.equal(step, plain + r)
    for out_dtype in (None, torch.float32):
        wide = hip_ops.gemm(x.t(), w, bias, residual=r.float(), out_dtype=out_dtype)
        assert ((wide.double() - exact_step).abs() <= 2 * slack + 2.0 ** -8 * (exact.abs() + exact_step.abs())).all()


@pytest.fixture()
def recorded(monkeypatch):
    """The launchers on host tensors with empty plan tables and a library that notes its launches."""
    import torch
    from test_attention_routes import RecordingLibrary
    from torch_mojo_backend.eager_kernels import hip_ops

    lib = RecordingLibrary(_ek().lib())
    monkeypatch.setattr(_ek(), "lib", lambda: lib)
    monkeypatch.setattr(hip_ops, "_stream", lambda: 0)
    monkeypatch.setattr(hip_ops, "require_hip", lambda *a: None)
    monkeypatch.setattr(hip_ops, "_GEMM_PLANS", {})
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    return lib


def _launch(recorded, *args, **kwargs):
    """(entry, sizes and flags, scratch) of the product's launch and of the copies in front of it."""
    from torch_mojo_backend.eager_kernels import hip_ops
    recorded.launched.clear()
    hip_ops.gemm(*args, **kwargs)
    seen = []
    for name, args in recorded.launched:
        scratch = args[-2] if name == "tmb_gemm_ws" else 0
        seen.append((name, args[4:18] if name.startswith("tmb_gemm") else (), scratch))
    return seen


@pytest.mark.parametrize("m,n,k", [(100, 104, 4096), (300, 1024, 8192), (512, 2048, 8192), (2048, 2048, 2048)])
def test_the_launch_of_a_product_does_not_depend_on_the_one_before(recorded, m, n, k):
    """Same sizes and strides, once on a 16-byte boundary and once off it: whichever came first."""
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    store = torch.zeros(m * k + 8, dtype=torch.bfloat16)
    assert store.data_ptr() % 16 == 0
    on, off = store[:m * k].view(m, k), store[1:m * k + 1].view(m, k)
    b = torch.zeros(k, n, dtype=torch.bfloat16)
    fresh = []
    for a in (on, off):
        hip_ops._GEMM_PLANS.clear()
        fresh.append(_launch(recorded, a, b))
    assert fresh[0] != fresh[1]
    for order in ((0, 1), (1, 0)):
        hip_ops._GEMM_PLANS.clear()
        for _ in range(2):
            for i in order:
                assert _launch(recorded, (on, off)[i], b) == fresh[i], (order, i)


def test_the_launch_of_an_epilogue_does_not_depend_on_the_plain_product_before(recorded):
    """A transposed A: the rings take it without an epilogue only."""
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    a, b = torch.zeros(2048, 2048).bfloat16().t(), torch.zeros(2048, 2048).bfloat16()
    gelu = dict(epilogue=_ek().EPI_GELU_ERF)
    alone = _launch(recorded, a, b, **gelu)
    hip_ops._GEMM_PLANS.clear()
    plain = _launch(recorded, a, b)
    assert plain != alone
    for _ in range(2):
        assert _launch(recorded, a, b, **gelu) == alone and _launch(recorded, a, b) == plain


def test_a_product_that_runs_whole_is_given_no_scratch(recorded):
    """A transposed A: one round of whole tiles takes the first, a split launch the second."""
    import torch
    for m, n, k, pitch in ((3072, 768, 2048, 3072), (3000, 768, 2048, 3072), (768, 768, 16384, 768)):
        a, b = torch.zeros(k, pitch).bfloat16()[:, :m].t(), torch.zeros(k, n).bfloat16()
        splits = route(m, n, k, ta=1, lda=pitch, workspace=PLENTY)[2]
        (name, _, scratch), = _launch(recorded, a, b)
        assert scratch == splits * m * n * 4 and (name == "tmb_gemm_ws") == (splits > 0), (m, n, k)
        residual = torch.zeros(m, n).bfloat16()
        (name, _, _), = _launch(recorded, a, b, residual=residual)
        assert name == "tmb_gemm_residual_ws"


def test_products_of_depth_64_stay_on_their_kernel_beyond_four_gigabytes():
    """It addresses a tile at a time; the rings' 32-bit offsets from the base end there."""
    for m in (8192, (1 << 25) - 128, 1 << 25, 1 << 26):
        for tb in (0, 1):
            assert route(m, 1024, 64, tb=tb)[0] == STREAM64, m
    assert route(1 << 25, 1024, 64, lda=1 << 23)[0] == STREAM64
    assert route(1 << 25, 1024, 64, residual=1)[0] == ANY


@pytest.mark.gpu
def test_depth_64_beyond_four_gigabytes_matches_float64():
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    m, n = 1 << 25, 128
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(m // 64, 64, generator=g, device="cuda").bfloat16().repeat(64, 1)
    a[-1000:] = torch.randn(1000, 64, generator=g, device="cuda").bfloat16()
    b = torch.randn(64, n, generator=g, device="cuda").bfloat16()
    got = hip_ops.gemm(a, b)
    rows = torch.cat([torch.arange(0, 300), torch.arange(m // 2 - 200, m // 2 + 200), torch.arange(m - 1200, m)]).cuda()
    want = a[rows].double() @ b.double()
    bound = 66 * 2.0 ** -24 * (a[rows].double().abs() @ b.double().abs()) + 1e-6 + 2.0 ** -8 * want.abs()
    assert ((got[rows].double() - want).abs() <= bound).all()


def test_fp32_products_with_long_rows_stay_on_the_matrix_cores():
    """Lane offsets are 32-bit within a tile: what counts is the tile's rows times the pitch, and beyond that the
    aligned kernel, which addresses in 64 bits, takes the product."""
    f32 = dict(dtype=_ek().F32, workspace=PLENTY)
    for k in (1 << 23, (1 << 23) + 1, 1 << 26):
        kernel, _, splits = route(4, 8, k, tb=1, **f32)
        assert kernel == F32 and splits > 1, k
    assert route(1 << 24, 64, 100, ta=1, a_aligned=0, **f32)[0] == F32
    kernel, _, splits = route(64, 64, 1 << 25, tb=1, **f32)
    assert kernel == F32_WIDE and splits > 1 and (1 << 25) % (4 * splits) == 0
    assert route(64, 64, (1 << 25) + 4, tb=1, **f32)[0] == F32_WIDE
    for k in (4096, 3004):           # (runs of K need not come out even)
        dense = route(64, 60, k, tb=1, dtype=f32["dtype"], workspace=PLENTY, a_aligned=0)
        assert route(64, 60, k, tb=1, lda=1 << 25, **f32) == (F32_WIDE, 0, dense[2]) and dense[2] > 1
    assert route(64, 64, 1 << 25, tb=1, dtype=_ek().F32) == (F32_WIDE, 0, 0)
    assert route(1 << 26, 64, 64, ta=1, **f32)[0] == F32_WIDE
    assert route(64, 64, 1 << 25, tb=1, residual=1, **f32) == _ek().ERR_UNSUPPORTED
    assert route(64, 64, 1 << 25, tb=1, a_aligned=0, **f32)[0] == SIMT     # (the launcher pads it first)


def test_long_runs_of_k_are_padded_for_the_aligned_kernels():
    """(m, n, k, transposed A, transposed B), A (the first two: and B) off a 16-byte boundary, whose padded copies measured
    1.3 .. 1.6 times as fast as the operands where they lie, some of them on a split launch; and a shape that stays."""
    ek = _ek()
    for m, n, k, ta, tb in ((597, 5159, 7235, 0, 1), (2336, 512, 8672, 0, 1), (192, 7168, 4704, 1, 0)):
        ask = ek.lib().tmb_gemm_in_place_workspace_bytes
        assert ask(1, m, n, k, m if ta else k, k if tb else n, 0, ta, ta, tb, 1, ek.BF16) == -1, (m, n, k)
        assert ask(1, 1999, 1001, 1500, 1999 if ta else 1500, 1500 if tb else 1001, 0, 0, ta, tb, 1, ek.BF16) == 0


def test_fp32_operands_that_no_matrix_kernel_reads_are_padded():
    """Fewer than four contiguous elements, or rows out of reach of 32-bit offsets; and where padding is only the faster
    way, the copies run on the kernel for which they are made."""
    pays = 0
    for m, n, k, ta, tb, extra in itertools.product((3, 4, 64, 65, 5000, 1 << 24, 1 << 25), (3, 4, 128, 129, 8000, 1 << 23),
                                                    (3, 4, 31, 33, 200, 1 << 23, 1 << 26), (0, 1), (0, 1), (0, 1 << 23)):
        lda, ldb = (m if ta else k) + extra, (k if tb else n) + extra
        pad = _ek().lib().tmb_gemm_f32_padding_pays(1, m, n, k, lda, ldb, 0, 0, ta, tb)
        lines, lanes = (32 if ta else min(m, 64)), (min(n, 128) if tb else 32)
        reach = (1 << 30) - 256
        read = (m if ta else k) >= 4 and (k if tb else n) >= 4 and lda < reach // max(lines - 1, 1) \
            and ldb < reach // max(lanes - 1, 1)
        if not read:
            assert pad == 1, (m, n, k, ta, tb, extra)
        elif pad and m * n < 1 << 31:
            depth = k if k % 4 == 0 else (k + 63) // 64 * 64
            assert route(m, n, depth, 0, 1, _ek().F32)[0] == F32_WIDE, (m, n, k, ta, tb, extra)
            pays += 1
    assert pays > 20


FORMS_F32 = [dict(ta=ta, tb=tb, a_aligned=a, b_aligned=b) for ta, tb, a, b in itertools.product((0, 1), repeat=4)]


@pytest.mark.parametrize("dtype_name", ["BF16", "F16", "F32"])
def test_short_k_over_many_tiles_leaves_the_kernels_whose_waves_share_k(dtype_name):
    """One slice of K or less for a workgroup's four waves and a launch of many tiles: the vector kernel or the 128 x 128
    one, as before those kernels; few tiles or a longer K stay, whatever the form."""
    dtype = getattr(_ek(), dtype_name)
    waves = F32 if dtype_name == "F32" else ANY
    many = [(48, 5222, 16, 8), (48, 402, 354, 8), (1, 6461, 1251, 9), (5, 2632, 758, 8)]
    for (batch, m, n, k), form in itertools.product(many, FORMS_F32):
        if dtype_name != "F32" and form["a_aligned"] and not form["ta"] and k % 8 == 0:
            form = dict(form, a_aligned=0)      # (aligned 16-bit operands have kernels of their own)
        got = route(m, n, k, batch=batch, dtype=dtype, **form)
        assert got in ((SIMT, 0, 0), (F32_WIDE, 0, 0)), (batch, m, n, k, form)
    for (batch, m, n, k), form in itertools.product([(1, 100, 200, 30), (1, 8, 8, 8), (1, 2000, 999, 150), (48, 401, 350, 130),
                                                     (1, 333, 77, 50), (2, 5000, 3001, 333)], FORMS_F32):
        form = dict(form, a_aligned=0)
        assert route(m, n, k, batch=batch, dtype=dtype, **form)[0] == waves, (batch, m, n, k, form)
    # the waves' kernels carry a residual, the others' product and the add apart where they are the faster way
    off = dict(a_aligned=0, dtype=dtype, residual=1)
    assert route(2000, 999, 150, **off)[0] == waves
    if dtype_name == "F32":
        for batch, m, n, k in ((1, 7016, 248, 12), (1, 840, 3000, 8), (5, 1696, 1848, 312)):
            assert route(m, n, k, tb=1, batch=batch, dtype=dtype) == (F32_WIDE, 0, 0)
        assert route(4104, 608, 8, tb=1, batch=48, **off) == _ek().ERR_UNSUPPORTED
        assert route(112, 6216, 8, tb=1, batch=48, residual=1, dtype=dtype) == _ek().ERR_UNSUPPORTED
        assert route(4096, 4096, 4096, residual=1, dtype=dtype) == _ek().ERR_UNSUPPORTED


@pytest.mark.gpu
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("ta,tb", itertools.product((False, True), repeat=2))
def test_short_k_over_many_tiles_matches_float64(dtype_name, ta, tb):
    """Ragged edges of the 64 x 64 and 128 x 128 tiles, with and without a residual, and (fp32, the last two) padded copies."""
    import torch
    from torch_mojo_backend.eager_kernels import EPI_GELU_TANH, hip_ops
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(7)
    for batch, m, n, k in ((48, 402, 354, 8), (48, 1100, 17, 9), (1, 6461, 1251, 9), (1, 3001, 3501, 61), (2, 2001, 2000, 97)):
        rows, cols = ((batch, k, m) if ta else (batch, m, k)), ((batch, n, k) if tb else (batch, k, n))
        off = torch.randn(batch * m * k + 1, generator=g, device="cuda").to(dtype)[1:].view(rows)
        a, b = (off.mT if ta else off), torch.randn(cols, generator=g, device="cuda").to(dtype)
        b = b.mT if tb else b
        if batch == 1:
            a, b = a[0], b[0]
        bias = torch.randn(n, generator=g, device="cuda").to(dtype)
        r = torch.randn(*a.shape[:-1], n, generator=g, device="cuda").to(dtype)
        a64, b64 = a.double().contiguous(), b.double().contiguous()
        exact = a64 @ b64 + bias.double()
        slack = (k + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + exact.abs() + r.double().abs()) + 1e-6
        ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
        plain = hip_ops.gemm(a, b, bias)
        assert ((plain.double() - exact).abs() <= slack + ulp * exact.abs()).all(), (batch, m, n, k)
        once = hip_ops.gemm(a, b, bias, residual=r)
        want = exact + r.double()
        # (product and sum may be rounded apart)
        assert ((once.double() - want).abs() <= slack + ulp * (exact.abs() + want.abs())).all(), (batch, m, n, k)
        assert torch.equal(hip_ops.gemm(a, b, bias, residual=r, round_like_unfused=True), plain + r)
        if dtype != torch.float32:
            assert torch.equal(hip_ops.gemm(a, b, bias, epilogue=EPI_GELU_TANH, round_like_unfused=True),
                               hip_ops.gelu(plain, "tanh"))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float32"])
@pytest.mark.parametrize("form", itertools.product((False, True), (False, True), (0, 1)))
def test_epilogues_rounded_like_separate_operations_have_their_bits(dtype_name, form):
    """Whatever the product runs on: small, split, ring, transposed A, any-layout, padded with and without its form, K = 64."""
    import torch
    from torch_mojo_backend.eager_kernels import EPI_GELU_ERF, EPI_GELU_TANH, hip_ops
    ta, tb, off = form
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(11)
    for m, n, k in ((256, 256, 256), (128, 768, 768), (2000, 768, 3072), (2049, 2048, 4096), (2048, 2304, 2049), (100, 100, 5001),
                    (4096, 2048, 64), (1999, 1001, 150), (597, 2001, 7235)):
        a = torch.randn(m * k + off, generator=g, device="cuda").to(dtype)[off:].view((k, m) if ta else (m, k))
        b = torch.randn((n, k) if tb else (k, n), generator=g, device="cuda").to(dtype)
        a, b = (a.t() if ta else a), (b.t() if tb else b)
        bias, r = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((n,), (m, n)))
        plain = hip_ops.gemm(a, b, bias)
        assert torch.equal(hip_ops.gemm(a, b, bias, residual=r, round_like_unfused=True), plain + r), (m, n, k)
        for epilogue, kind in ((EPI_GELU_TANH, "tanh"), (EPI_GELU_ERF, "none")):
            got = hip_ops.gemm(a, b, bias, epilogue=epilogue, round_like_unfused=True)
            assert torch.equal(got, hip_ops.gelu(plain, kind)), (m, n, k, kind)
            got = hip_ops.gemm(a, b, bias, epilogue=epilogue, residual=r, round_like_unfused=True)
            assert torch.equal(got, hip_ops.gelu(plain, kind) + r), (m, n, k, kind)


def test_the_launcher_pads_fp32_operands_of_short_k(recorded):
    """Off a 16-byte boundary; the copies run without a residual, which is added apart."""
    import torch
    m, n, k = 6000, 7000, 96
    store, b = torch.zeros(m * k + 4), torch.zeros(k, n)
    off, residual = store[1:m * k + 1].view(m, k), torch.zeros(m, n)
    for kw in ({}, {"residual": residual}):
        assert [name for name, _, _ in _launch(recorded, off, b, **kw)] == ["tmb_pad_rows", "tmb_gemm"]
    assert [name for name, _, _ in _launch(recorded, off[:300], b[:, :400])] == ["tmb_gemm"]


@pytest.mark.gpu
@pytest.mark.parametrize("case", [
    # (m, n, k, pitch of A, A stored [K, M])
    (4, 8, (1 << 23) + 1, None, False),      # long rows, few of them
    (64, 60, 4096, 1 << 25, False),          # rows out of reach: the wide kernel, K split
    (64, 60, 3004, 1 << 25, False),          # and in runs that do not come out even
    (130, 60, 100, 35651584, True)])         # k-rows out of reach
def test_fp32_long_rows_match_float64(case):
    import torch
    from torch_mojo_backend.eager_kernels import hip_ops
    m, n, k, pitch, ta = case
    g = torch.Generator(device="cuda").manual_seed(m)
    rows, cols = (k, m) if ta else (m, k)
    if pitch is None:
        stored = torch.randn(rows, cols, generator=g, device="cuda")
    else:
        stored = torch.empty((rows - 1) * pitch + cols, device="cuda").as_strided((rows, cols), (pitch, 1))
        stored.copy_(torch.randn(rows, cols, generator=g, device="cuda"))
    a = stored.t() if ta else stored
    b = torch.randn(n, k, generator=g, device="cuda").t()
    bias = torch.randn(n, generator=g, device="cuda")
    got = hip_ops.gemm(a, b, bias)
    exact, size = bias.double().expand(m, n).clone(), bias.double().abs().expand(m, n).clone()
    for at in range(0, k, 1 << 18):
        x, y = a[:, at:at + (1 << 18)].double().contiguous(), b[at:at + (1 << 18)].double().contiguous()
        exact += x @ y
        size += x.abs() @ y.abs()
    # k roundings in a chain would be k 2^-24 of the sum of magnitudes; runs of at most 2^19 of them are chained
    assert ((got.double() - exact).abs() <= (min(k, 1 << 19) + 40) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("batch,m,n,k,ta,tb,kernel", [
    (24, 32, 50304, 16, 0, 0, F32_WIDE),     # 77 us, 112 on 32 x 32 tiles
    (4, 32, 50257, 16, 1, 1, F32_WIDE),      # 20 and 24 (a padded B)
    (25, 2208, 16, 16, 0, 0, F32_WIDE),      # 6.5 and 8.3
    (57, 192, 7104, 144, 1, 0, F32_WIDE),    # 358 and 485
    (13, 160, 50304, 176, 1, 1, F32_WIDE),   # 597 and 648
    (1, 4560, 50257, 37, 1, 1, SIMT),        # 587 and 826
    (1, 4528, 50257, 40, 0, 0, SIMT)])       # 576 and 840
def test_fp32_products_of_short_k_over_many_tiles_run_where_they_are_fastest(batch, m, n, k, ta, tb, kernel):
    """The many small tiles of the waves-share-K kernel cost as much as their bytes there."""
    aligned = kernel == F32_WIDE
    assert route(m, n, k, ta, tb, _ek().F32, batch=batch, a_aligned=aligned, b_aligned=aligned)[0] == kernel
