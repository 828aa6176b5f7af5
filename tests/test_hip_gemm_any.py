"""GPU parity of the kernel that takes 16-bit operands of any layout and alignment where they lie: its
tiles, tile and K edges, bases off a 16-byte boundary, every layout, its epilogue and its split launch;
and the rule that chooses between it and padded copies, over all forms on the CPU."""

import itertools

import pytest
import torch

from helpers import ULP

HALF = [torch.bfloat16, torch.float16]


def _ops():
    from torch_mojo_backend.eager_kernels import hip_ops
    return hip_ops


def _operand(rows, cols, transposed, off, pitch, gen, dtype, batch=None):
    """[.., rows, cols], stored transposed or not, `off` elements behind an aligned base, `pitch` more
    elements between rows; what lies between is NaN."""
    r, c = (cols, rows) if transposed else (rows, cols)
    n = 1 if batch is None else batch
    store = torch.full((n * r * (c + pitch) + off + 64,), float("nan"), device="cuda").to(dtype)
    t = store[off:off + n * r * (c + pitch)].view(n, r, c + pitch)[:, :, :c]
    t.copy_(torch.randn(n, r, c, generator=gen, device="cuda"))
    t = t if batch is not None else t[0]
    return t.transpose(-1, -2) if transposed else t


def _check(got, a, b, extra64, what):
    """|got - exact| <= half a unit of the result's type plus the float32 accumulation bound."""
    a64, b64 = a.double().contiguous(), b.double().contiguous()
    exact = a64 @ b64 + extra64
    bound = (a.shape[-1] + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + exact.abs()) + 1e-6
    err = (got.double() - exact).abs()
    assert (err <= bound + ULP[got.dtype] * exact.abs()).all(), (what, (err - bound).max().item())


# (m, n, k): the smallest it takes, one per tile, ragged everywhere, K of one slice, K that leaves waves
# without one, K long enough to be split
SHAPES = [(8, 8, 8), (9, 15, 11), (1, 67, 129), (17, 33, 65), (40, 3001, 511), (250, 300, 1000), (231, 361, 343),
          (333, 999, 77), (1999, 1001, 150), (100, 100, 5001), (13, 93, 3075), (65, 129, 63), (1999, 1001, 1500)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("ta,tb", itertools.product([False, True], [False, True]))
def test_any_layout_and_alignment_matches_float64(mnk, dtype, ta, tb):
    m, n, k = mnk
    g = torch.Generator(device="cuda").manual_seed(m + 3 * n + 7 * k)
    bias = torch.randn(n + 1, generator=g, device="cuda").to(dtype)[1:]
    for off, pitch in ((0, 0), (1, 0), (3, 5)):
        a = _operand(m, k, ta, off, pitch, g, dtype)
        b = _operand(k, n, tb, off, pitch, g, dtype)
        _check(_ops().gemm(a, b, bias), a, b, bias.double(), (mnk, off, pitch))
        _check(_ops().gemm(a, b), a, b, 0.0, (mnk, off, pitch))


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", itertools.product([False, True], [False, True]))
def test_any_layout_batches_epilogue_and_residual(ta, tb):
    dtype, ops = torch.bfloat16, _ops()
    from torch_mojo_backend.eager_kernels import EPI_GELU_TANH
    g = torch.Generator(device="cuda").manual_seed(5)
    a, b = _operand(33, 77, ta, 1, 3, g, dtype, 5), _operand(77, 65, tb, 0, 1, g, dtype, 5)
    _check(ops.gemm(a, b), a, b, 0.0, "batched")
    for m, n, k in ((50, 121, 131), (30, 70, 5001)):    # one launch; split along K
        a, b = _operand(m, k, ta, 1, 2, g, dtype), _operand(k, n, tb, 1, 0, g, dtype)
        bias = torch.randn(n, generator=g, device="cuda").to(dtype)
        res = torch.randn(m, n, generator=g, device="cuda")
        wide = ops.gemm(a, b, bias, residual=res, out_dtype=torch.float32)
        _check(wide, a, b, bias.double() + res.double(), "float32 residual and result")
        plain = ops.gemm(a, b, bias)
        # rounded step by step: exactly the separate operations' results
        step = ops.gemm(a, b, bias, residual=res.to(dtype), round_like_unfused=True)
        assert torch.equal(step, plain + res.to(dtype))
        fused = ops.gemm(a, b, bias, epilogue=EPI_GELU_TANH, round_like_unfused=True)
        assert torch.equal(fused, ops.gelu(plain, "tanh"))


def test_choice_between_in_place_and_padded_on_the_host():
    from torch_mojo_backend import eager_kernels as ek

    ask = ek.lib().tmb_gemm_in_place_workspace_bytes
    for ta, tb, aa, ba, plain, dt in itertools.product((0, 1), (0, 1), (0, 1), (0, 1), (0, 1), (ek.BF16, ek.F16)):
        for m, n, k in itertools.product((1, 8, 1001, 50257), (8, 77, 50257), (8, 750, 30001)):
            lda, ldb = (m if ta else k), (k if tb else n)
            ws = ask(1, m, n, k, lda, ldb, aa, ba, ta, tb, plain, dt)
            if ta and m < 8:
                assert ws == -1      # fewer than eight contiguous elements: not read in place
            elif ws >= 0:
                assert ws % (4 * m * n) == 0 and ws // (4 * m * n) <= 16
        # small products are read in place whatever their form; large ones are not worth it
        assert ask(1, 100, 200, 300, 100 if ta else 300, 300 if tb else 200, aa, ba, ta, tb, plain, dt) >= 0
        assert ask(1, 16385, 16385, 16385, 16385, 16385, aa, ba, ta, tb, plain, dt) == -1
    assert ask(1, 100, 200, 300, 300, 200, 0, 0, 0, 0, 1, ek.F32) == -1
    assert ask(1, 0, 200, 300, 300, 200, 0, 0, 0, 0, 1, ek.BF16) == -1
