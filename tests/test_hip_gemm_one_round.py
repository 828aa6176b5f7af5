"""GPU parity of the 64-deep ring tiles that run in one round of the CUs: products on both sides of the rules that choose
them, with partial tiles, the fewest stages the rings take, every operand layout, epilogue, batches and narrow outputs."""

import pytest
import torch

from test_hip_gemm_small import HALF, _check, _inputs, _ops

pytestmark = pytest.mark.gpu


def _ek():
    from torch_mojo_backend import eager_kernels as ek
    return ek

# (m, n, k): 64 x 128 tiles in one round (two of them with one row or column past a tile), 128 x 128 in one round, 64 x 128
# two to a CU in one round and in more, products that no longer split, runs of a split on eight waves, narrow outputs of few
# and many rows, and 64 x 64 tiles whose waves share K
ROW_MAJOR = [(2049, 768, 256), (2048, 776, 320), (4096, 1024, 256), (3400, 1160, 320), (5400, 768, 256), (6785, 776, 320),
             (2113, 768, 2304), (2700, 768, 3072), (520, 1096, 8192), (300, 64, 4160), (32768, 48, 256), (32709, 56, 320),
             (1025, 1000, 256), (960, 776, 3072)]
TRANSPOSED = [(768, 768, 256), (1416, 840, 320), (3072, 768, 2048), (2056, 2048, 576), (1408, 840, 4160)]


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", ROW_MAJOR)
@pytest.mark.parametrize("trans_b", [False, True])
def test_row_major_products_match_float64(mnk, dtype, trans_b):
    a, b, bias, _ = _inputs(*mnk, dtype, trans_b)
    _check(_ops().gemm(a, b, bias), a, b, bias.double(), mnk)
    _check(_ops().gemm(a, b), a, b, 0.0, mnk)


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", TRANSPOSED)
def test_transposed_products_match_float64(mnk, dtype):
    m, n, k = mnk
    a, b, _, _ = _inputs(k, n, m, dtype, True)      # [k, m] and [n, m]: the second one only sets the generator's course
    b = torch.randn(k, n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(k)).to(dtype)
    _check(_ops().gemm(a.t(), b), a.t().contiguous(), b, 0.0, mnk)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("mnk", [(2049, 776, 320), (4001, 1000, 256), (5400, 776, 256), (1025, 1000, 256), (33000, 40, 256)])
def test_epilogues_residuals_and_batches(mnk, trans_b):
    a, b, bias, g = _inputs(*mnk, torch.bfloat16, trans_b)
    rounded = _ops().gemm(a, b, bias)
    for kind, epilogue in (("tanh", _ek().EPI_GELU_TANH), ("none", _ek().EPI_GELU_ERF)):
        got = _ops().gemm(a, b, bias, epilogue, round_like_unfused=True)
        assert torch.equal(got, _ops().gelu(rounded, kind)), (mnk, kind)
    r = torch.randn(*mnk[:2], generator=g, device="cuda").bfloat16()
    assert torch.equal(_ops().gemm(a, b, bias, residual=r, round_like_unfused=True), rounded + r)
    m, n, k = mnk[0] // 5, mnk[1], mnk[2]
    a, b, _, _ = _inputs(m, n, k, torch.bfloat16, trans_b, batch=5)
    _check(_ops().gemm(a, b), a, b, 0.0, (5, m, n, k))


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("mnk", [(2049, 768, 264), (2048, 776, 1000), (3400, 1160, 312), (5400, 768, 328), (6785, 776, 2008),
                                 (1203, 1024, 2000), (12500, 2304, 280), (65, 9000, 4088)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_k_that_ends_inside_a_stage(mnk, dtype, trans_b):
    """The last stage holds zeros past the end of K, whatever lies there: a row's neighbour starts with an infinity."""
    a, b, bias, _ = _inputs(*mnk, dtype, trans_b)
    a[7, 0] = float("inf")
    a[11, mnk[2] - 1] = float("nan")
    got = _ops().gemm(a, b, bias)
    bad = ~got.isfinite()
    assert bad[7].all() and bad[11].all() and bad.sum() == 2 * mnk[1]
    a[7, 0] = a[11, mnk[2] - 1] = 0
    got[7] = got[11] = 0
    bias64 = bias.double().expand(mnk[0], -1).clone()
    a[7] = a[11] = 0
    bias64[7] = bias64[11] = 0
    _check(got, a, b, bias64, mnk)


@pytest.mark.parametrize("dtype", HALF)
@pytest.mark.parametrize("k", [2048, 2496, 4096])
def test_transposed_products_are_summed_in_short_chains(k, dtype):
    """2^29 first and its negative last, ones between. Float32 numbers of 2^29 lie 64 apart, more than what an MFMA adds at a
    time: one chain over K loses all the ones, chains of 512 lose those of the first and the last."""
    a, b = (torch.ones(k, n, device="cuda", dtype=dtype) for n in (3072, 768))
    a[0], a[-1], b[0], b[-1] = 2.0 ** 15, -2.0 ** 15, 2.0 ** 14, 2.0 ** 14
    got = _ops().gemm(a.t(), b)
    assert got.min() >= (k - 1024) * (1 - 2.0 ** -8) and got.max() <= k
