"""GPU parity of the fp32 kernel whose waves share K: every tile, all four operand layouts, extents
that end inside a 16-byte piece in either direction, operands at any 4-byte address inside memory
full of NaN, runs of K split over workgroups, and the residual epilogue."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from torch_mojo_backend.eager_kernels import hip_ops
    return hip_ops


def _embedded(rows, cols, seed, batch=None):
    """A matrix at an odd offset inside a buffer of NaN, row pitch cols + 3."""
    lead = () if batch is None else (batch,)
    g = torch.Generator(device="cuda").manual_seed(seed)
    buf = torch.full((*lead, rows + 2, cols + 3), float("nan"), device="cuda")
    buf[..., 1:rows + 1, 1:cols + 1] = torch.randn(*lead, rows, cols, generator=g, device="cuda")
    return buf[..., 1:rows + 1, 1:cols + 1]


def _check(got, a, b, extra, what):
    """|got - exact| <= the a-priori bound of k float32 multiply-adds."""
    a64, b64 = a.double(), b.double().contiguous()
    exact = a64 @ b64 + extra
    bound = (a.shape[-1] + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + exact.abs()) + 1e-6
    assert ((got.double() - exact).abs() <= bound).all(), what


# (m, n, k): one, two and three elements past a piece, the smallest extents, runs of K that are split, and (the last seven)
# one per tile: 32 x 32 with fp32 products over many rounds, 32 x 32 with eight and four waves, 32 x 64, 64 x 64 with four
# and eight waves, and one of these split
SHAPES = [(40, 70, 33), (500, 1000, 130), (777, 1025, 259), (1332, 770, 770), (750, 2306, 260), (4, 4, 4), (5, 6, 7), (33, 129, 35),
          (65, 34, 62), (130, 770, 3001), (31, 67, 12565),
          (501, 1001, 101), (101, 203, 150), (161, 1367, 133), (877, 573, 683), (1571, 1139, 243), (823, 1135, 163),
          (37, 2179, 2363)]


@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
def test_any_extent_pitch_and_layout(mnk, trans_a, trans_b):
    m, n, k = mnk
    a = _embedded(k, m, 1).t() if trans_a else _embedded(m, k, 1)
    b = _embedded(n, k, 2).t() if trans_b else _embedded(k, n, 2)
    bias = torch.randn(n, device="cuda")
    _check(_ops().gemm(a, b, bias), a, b, bias.double(), mnk)
    res = _embedded(m, n, 3)
    _check(_ops().gemm(a, b, bias, residual=res), a, b, bias.double() + res.double(), mnk)


def test_batches_and_extents_below_one_piece():
    a, b = _embedded(37, 30, 4, batch=5), _embedded(30, 41, 5, batch=5)
    _check(_ops().gemm(a, b), a, b, 0.0, "batched")
    for m, n, k in ((3, 5, 9), (9, 3, 5), (5, 9, 3), (1, 1, 1)):   # the any-layout kernel
        a, b = _embedded(m, k, 6), _embedded(k, n, 7)
        _check(_ops().gemm(a, b), a, b, 0.0, (m, n, k))
        _check(_ops().gemm(a.t().contiguous().t(), b.t().contiguous().t()), a, b, 0.0, (m, n, k))


def test_the_result_does_not_depend_on_alignment():
    """Pieces that end at an edge are read shifted: same values, same order of the sums."""
    a, b = _embedded(100, 75, 8), _embedded(90, 75, 9).t()
    want = _ops().gemm(a, b)
    assert torch.equal(_ops().gemm(a.contiguous(), b.t().contiguous().t()), want)
