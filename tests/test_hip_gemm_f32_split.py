"""fp32 products on the bf16 matrix cores: as exact as fp32 products over the whole range of fp32, infinities and NaN
where they belong, and every edge of the 128 x 128 kernel (rows, columns, the last stage of K, runs of K split over
workgroups, operands off 16-byte boundaries)."""

import itertools

import pytest
import torch

from test_gemm_routes import F32, F32_WIDE, PLENTY, route


def _ops():
    from torch_mojo_backend.eager_kernels import hip_ops
    return hip_ops


def _operand(rows, cols, stored_transposed, seed, offset=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r, c = (cols, rows) if stored_transposed else (rows, cols)
    buf = torch.full((r * c + offset,), float("nan"), device="cuda")
    x = buf[offset:].view(r, c)
    x.copy_(torch.randn(r, c, generator=g, device="cuda").double() * scale)
    return x.t() if stored_transposed else x


def _check(got, a, b, extra=0.0):
    """|got - exact| <= the a-priori bound of k float32 multiply-adds; among subnormals each of up to 16 partial sums is
    rounded to a multiple of the smallest one."""
    a64, b64 = a.double().contiguous(), b.double().contiguous()
    exact = a64 @ b64 + extra
    bound = (a.shape[-1] + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + exact.abs()) + 8 * 2.0 ** -149
    assert ((got.double() - exact).abs() <= bound).all()


# whole tiles, one row / column past them, K that ends inside a stage or a 16-byte piece; the last two split
WIDE = [(1408, 2304, 768), (1409, 2433, 772), (2047, 2300, 132), (3001, 1030, 515), (750, 768, 3072), (385, 770, 8201)]


def test_the_shapes_reach_the_kernel():
    from torch_mojo_backend import eager_kernels as ek
    for m, n, k in WIDE:
        for ta, tb in itertools.product((0, 1), repeat=2):
            aligned = (m if ta else k) % 4 == 0 and (k if tb else n) % 4 == 0
            if aligned or k >= 512:
                kernel, _, splits = route(m, n, k, ta, tb, ek.F32, a_aligned=aligned, b_aligned=aligned, workspace=PLENTY)
                assert kernel == F32_WIDE and (splits > 0) == (m < 1000), (m, n, k, ta, tb)
    assert route(300, 500, 300, dtype=ek.F32, workspace=PLENTY)[0] == F32


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", WIDE)
@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
def test_edges_of_the_128_tile(mnk, trans_a, trans_b):
    m, n, k = mnk
    bias = torch.randn(n, device="cuda")
    for offset in (0, 1):
        a, b = _operand(m, k, trans_a, 1, offset), _operand(k, n, trans_b, 2, offset)
        _check(_ops().gemm(a, b, bias), a, b, bias.double())


# the kernel whose waves share K, at any layout and alignment: fp32 products (K <= 128) in one round of tiles and in several,
# 32 x 32 tiles with eight waves (one round), split, and with four, 32 x 64, 64 x 64 with four and with eight, split
SHARED = [(300, 500, 100), (1000, 2000, 128), (300, 500, 300), (64, 128, 2000), (1788, 132, 136), (260, 1764, 680),
          (1776, 1072, 252), (1040, 936, 152), (132, 1672, 1184)]


def _kernels_of(shapes, **alignment):
    """{(tile, fp32 products, split, all tiles in one round)} of the products on the kernel whose waves share K."""
    from torch_mojo_backend import eager_kernels as ek
    took = set()
    for (m, n, k), ta, tb in itertools.product(shapes, (0, 1), (0, 1)):
        kernel, tile, splits = route(m, n, k, ta, tb, ek.F32, workspace=PLENTY, **alignment)
        if kernel == F32:
            rounds = -(-m // 32) * -(-n // 32) * max(splits, 1) / 256
            took.add((tile, k <= 128, splits > 0, tile > 0 or rounds <= 1))
    return took


def test_the_shapes_take_every_tile_with_either_product():
    """A refit of the models' constants must not drop one (32 x 32 tiles have eight waves where they run in one round)."""
    import test_hip_gemm_f32_edges
    every = {(0, True, False, True), (0, True, False, False), (0, False, False, True), (0, False, True, True),
             (0, False, False, False), (1, False, False, True), (2, False, False, True), (3, False, False, True),
             (3, False, True, True)}
    unaligned = dict(a_aligned=0, b_aligned=0)
    assert _kernels_of(SHARED) >= every and _kernels_of(SHARED, **unaligned) >= every
    assert _kernels_of(test_hip_gemm_f32_edges.SHAPES, **unaligned) >= every


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", WIDE + SHARED)
@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
def test_a_product_that_stands_alone_is_rounded_once(mnk, trans_a, trans_b):
    """One nonzero of 24 bits in each row: the large part of the product is exact, the sum of the small ones (2^-6.9 of
    it) rounded seven times to 2^-23 of itself, and their sum once: 2^-24 (1 + 1/4). Without the partial products of
    middle and low part, or with all in one sum, rows are off by three times that; without the low parts by 2^7."""
    m, n, k = mnk
    for offset in (0, 1):
        g = torch.Generator(device="cuda").manual_seed(11)
        where = torch.randint(0, k, (m, 1), generator=g, device="cuda")
        where[0], where[-1] = k - 1, k // 32 * 32 - 1     # (the last k, and the last of the stages that are whole)
        a = _operand(m, k, trans_a, 12, offset)
        kept = a.gather(1, where)
        a.zero_().scatter_(1, where, kept)
        b = _operand(k, n, trans_b, 13, offset)
        exact = kept.double() * b[where.flatten()].double()
        assert ((_ops().gemm(a, b).double() - exact).abs() <= 1.25 * 2.0 ** -24 * exact.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", WIDE + SHARED)
@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
def test_dense_operands_keep_all_three_parts(mnk, trans_a, trans_b):
    """Root mean square error of normal operands. n additions of equal weight, each rounded by 0.6 * 2^-24 of what has
    been summed, leave 0.6 * 2^-24 * sqrt(n / 2): n is K for fp32 products (128 here at most, 2.8e-7) and K / 32
    otherwise (8201: 4.1e-7). Without the low parts the error is 2^-18 of the result and more."""
    m, n, k = mnk
    a, b = _operand(m, k, trans_a, 14, 1), _operand(k, n, trans_b, 15, 1)
    exact = a.double().contiguous() @ b.double().contiguous()
    assert (_ops().gemm(a, b).double() - exact).norm() <= 5e-7 * exact.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(1408, 2304, 768), (300, 500, 300), (64, 128, 2000)])
@pytest.mark.parametrize("scales", [(2.0 ** -130, 2.0 ** 60), (2.0 ** -118, 2.0 ** -10), (2.0 ** 115, 2.0 ** -60),
                                    (2.0 ** 100, 2.0 ** 10), (1.0, 2.0 ** -149)])
def test_the_ends_of_the_range(mnk, scales):
    """Subnormal operands and results, and operands and results too large for the factor that the split is given room
    with: as exact as any (operands are rounded to float32 before, so what they are is what is multiplied)."""
    m, n, k = mnk
    a, b = _operand(m, k, False, 3, scale=scales[0]), _operand(k, n, True, 4, scale=scales[1])
    _check(_ops().gemm(a, b), a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(1408, 2304, 768), (300, 500, 300), (64, 128, 2000), (750, 768, 3072)])
def test_infinities_and_nan(mnk):
    """Each as in the float64 product of the same operands; rows and columns without them are not touched."""
    m, n, k = mnk
    a, b = _operand(m, k, False, 5), _operand(k, n, True, 6)
    a[3, 7], a[m - 2, 0], a[m // 2, k - 1] = float("inf"), float("nan"), float("-inf")
    b[k // 2, 5], b[7, n - 1] = float("inf"), 0.0
    got, exact = _ops().gemm(a, b), a.double() @ b.double().contiguous()
    assert torch.equal(got.isnan(), exact.isnan()) and torch.equal(got.isinf(), exact.isinf())
    assert torch.equal(got[got.isinf()], exact[exact.isinf()].float())
    rows = torch.ones(m, dtype=torch.bool)
    rows[[3, m - 2, m // 2]] = False
    columns = torch.ones(n, dtype=torch.bool)
    columns[5] = False
    _check(got[rows][:, columns], a[rows], b[:, columns])


def _spoil(a, b):
    """Infinities and a NaN in three rows of a, an infinity and a number without room for the factor in two columns of b
    (2^120: its products, below 2^123 for normal operands, and their sums are finite in float32 too); what is left of rows
    and columns."""
    m, k, n = a.shape[-2], a.shape[-1], b.shape[-1]
    a[..., 3, 7], a[..., m - 2, 0], a[..., m // 2, k - 1] = float("inf"), float("nan"), float("-inf")
    b[..., k // 2, 5], b[..., k - 2, n - 1] = float("inf"), 2.0 ** 120
    rows, columns = torch.ones(m, dtype=torch.bool), torch.ones(n, dtype=torch.bool)
    rows[[3, m - 2, m // 2]] = False
    columns[[5, n - 1]] = False
    return rows, columns


def _check_spoiled(a, b):
    clean = _ops().gemm(a, b)
    rows, columns = _spoil(a, b)
    got, exact = _ops().gemm(a, b), a.double() @ b.double().contiguous()
    assert torch.equal(got.isnan(), exact.isnan()) and torch.equal(got.isinf(), exact.isinf())
    assert torch.equal(got[got.isinf()], exact[exact.isinf()].float())
    assert torch.equal(got[..., rows, :][..., columns], clean[..., rows, :][..., columns])


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", WIDE + SHARED)
@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
def test_rows_and_columns_do_not_change_with_what_their_neighbours_hold(mnk, trans_a, trans_b):
    """Infinities and NaN spread as in the float64 product, whatever the layout and alignment, and rows and columns
    without them keep their bits."""
    m, n, k = mnk
    for offset in (0, 1):
        _check_spoiled(_operand(m, k, trans_a, 16, offset), _operand(k, n, trans_b, 17, offset))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(3, 700, 1100, 260), (5, 130, 70, 201)])
def test_batches_do_not_change_with_what_their_neighbours_hold(shape):
    batch, m, n, k = shape
    a = torch.stack([_operand(m, k, False, 18 + i) for i in range(batch)])
    b = torch.stack([_operand(k, n, False, 28 + i) for i in range(batch)])
    clean = _ops().gemm(a, b)
    _spoil(a[1], b[1])
    got = _ops().gemm(a, b)
    assert torch.equal(got[0], clean[0]) and torch.equal(got[2:], clean[2:])
    _check_spoiled(a[2:3].clone(), b[2:3].clone())
    assert torch.equal(_ops().gemm(a[1:2], b[1:2]).isnan(), got[1:2].isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(1408, 2304, 768), (300, 500, 300), (64, 128, 2000)])
def test_results_beyond_the_factors_room_leave_their_neighbours_alone(mnk):
    """Finite rows of 2^100, whose sums the split has no room for: as exact as any, and other rows keep their bits."""
    m, n, k = mnk
    a, b = _operand(m, k, False, 19), _operand(k, n, True, 20)
    clean = _ops().gemm(a, b)
    a[5] *= 2.0 ** 100
    got = _ops().gemm(a, b)
    _check(got, a, b)
    others = [r for r in range(m) if r != 5]
    assert torch.equal(got[others], clean[others])


@pytest.mark.gpu
@pytest.mark.parametrize("mnk", [(750, 768, 3072), (385, 770, 8201), (1408, 2304, 768)])
def test_a_residual_has_the_bits_of_product_and_sum(mnk):
    """Carried by the reduction of a split launch, added by the caller otherwise."""
    m, n, k = mnk
    a, b, bias = _operand(m, k, False, 7), _operand(k, n, True, 8), torch.randn(n, device="cuda")
    r = _operand(m, n, False, 9)
    assert torch.equal(_ops().gemm(a, b, bias, residual=r), _ops().gemm(a, b, bias) + r)
