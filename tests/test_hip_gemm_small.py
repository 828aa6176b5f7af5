"""GPU parity of the kernel for small 16-bit products (few rows, or tiles that fit one round of the
CUs): every tile it has, tile edges, K slices that do not fill a wave, both layouts of B, and its
epilogue in both rounding modes."""

import pytest
import torch

from helpers import ULP

pytestmark = pytest.mark.gpu

HALF = [torch.bfloat16, torch.float16]


def _ops():
    from torch_mojo_backend.eager_kernels import hip_ops
    return hip_ops


def _inputs(m, n, k, dtype, trans_b, batch=None):
    g = torch.Generator(device="cuda").manual_seed(m + 3 * n + 7 * k)
    lead = () if batch is None else (batch,)
    a = torch.randn(*lead, m, k, generator=g, device="cuda").to(dtype)
    b = torch.randn(*lead, *((n, k) if trans_b else (k, n)), generator=g, device="cuda").to(dtype)
    return a, (b.transpose(-1, -2) if trans_b else b), torch.randn(n, generator=g, device="cuda").to(dtype), g


def _check(got, a, b, extra64, what):
    """|got - exact| <= half a unit of the result's type plus the float32 accumulation bound."""
    a64, b64 = a.double(), b.double().contiguous()
    exact = a64 @ b64 + extra64
    bound = (a.shape[-1] + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + exact.abs()) + 1e-6
    err = (got.double() - exact).abs()
    assert (err <= bound + ULP[got.dtype] * exact.abs()).all(), (what, (err - bound).max().item())


# (m, n, k): one per tile of the kernel (16 x 16 .. 64 x 64), then edges: one row, one slice and a
# part of one, K below the waves' share, ragged rows and columns, the most tiles and the longest K
SHAPES = [(16, 768, 768), (128, 768, 3072), (128, 1024, 1024), (231, 2304, 768), (200, 2304, 768),
          (1024, 1024, 768), (1, 8, 8), (1, 50264, 72), (16, 4104, 4096), (17, 40, 520), (33, 72, 1000),
          (65, 136, 64), (255, 264, 4096), (1023, 1000, 264), (300, 768, 4096)]


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
def test_small_products_match_float64(mnk, dtype, trans_b):
    m, n, k = mnk
    a, b, bias, _ = _inputs(m, n, k, dtype, trans_b)
    _check(_ops().gemm(a, b, bias), a, b, bias.double(), mnk)
    _check(_ops().gemm(a, b), a, b, 0.0, mnk)


@pytest.mark.parametrize("dtype", HALF)
def test_small_products_ragged_columns_batches_and_row_pitches(dtype):
    a, b, bias, _ = _inputs(37, 1001, 200, dtype, True)    # N odd: K-major B only
    _check(_ops().gemm(a, b, bias), a, b, bias.double(), "odd columns")
    a, b, _, _ = _inputs(33, 64, 96, dtype, False, batch=5)
    _check(_ops().gemm(a, b), a, b, 0.0, "batched")
    a, b, bias, _ = _inputs(50, 120, 128, dtype, True)
    wide = torch.zeros(50, 200, dtype=dtype, device="cuda")
    wide[:, 8:136] = a
    assert torch.equal(_ops().gemm(wide[:, 8:136], b, bias), _ops().gemm(a, b, bias))


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", [(5, 1001, 768), (100, 768, 3072), (130, 768, 768), (300, 768, 4096), (2000, 768, 3072),
                                 (2000, 768, 5120)])
def test_small_epilogues(mnk, dtype):
    """Residual (storage type and float32) and GELU; the last two shapes run in one round of ring tiles and split along K."""
    m, n, k = mnk
    a, b, bias, g = _inputs(m, n, k, dtype, True)
    b = (b * 0.1)
    r32 = torch.randn(m, n, generator=g, device="cuda") * 3
    res = r32.to(dtype)
    plain = _ops().gemm(a, b, bias)
    for r in (res, r32):
        for out_dtype in (None, torch.float32):
            got = _ops().gemm(a, b, bias, residual=r, out_dtype=out_dtype)
            assert got.dtype == (out_dtype or dtype)
            _check(got, a, b, bias.double() + r.double(), (mnk, r.dtype, out_dtype))
    assert torch.equal(_ops().gemm(a, b, bias, residual=res, round_like_unfused=True), plain + res)
    from torch_mojo_backend import eager_kernels as ek
    for epi, approximate in ((ek.EPI_GELU_TANH, "tanh"), (ek.EPI_GELU_ERF, "none")):
        twice = _ops().gemm(a, b, bias, epilogue=epi, round_like_unfused=True)
        assert torch.equal(twice, _ops().gelu(plain, approximate))
        both = _ops().gemm(a, b, bias, epilogue=epi, residual=res, round_like_unfused=True)
        assert torch.equal(both, _ops().gelu(plain, approximate) + res)
        once = _ops().gemm(a, b, bias, epilogue=epi)
        exact = torch.nn.functional.gelu(a.double() @ b.double().contiguous() + bias.double(), approximate=approximate)
        slack = 1.2 * k * 2.0 ** -24 * (a.double().abs() @ b.double().abs().contiguous()) + 4e-6
        assert ((once.double() - exact).abs() <= slack + (ULP[dtype] + 1e-5) * exact.abs()).all()


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", [(231, 3072, 768), (300, 2304, 768), (1025, 1000, 256), (960, 776, 3072)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_a_16_bit_result_is_the_float32_result_rounded(mnk, dtype, trans_b):
    """The largest tile: the type of the result chooses neither the kernel nor the order of its sums."""
    a, b, bias, _ = _inputs(*mnk, dtype, trans_b)
    zero = torch.zeros(*mnk[:2], device="cuda")
    wide = _ops().gemm(a, b, bias, residual=zero, out_dtype=torch.float32)
    assert torch.equal(_ops().gemm(a, b, bias), wide.to(dtype))
