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
    assert route(100, 77, 50, a_aligned=0)[0] == ANY
    assert route(8192, 4096, 64)[0] == STREAM64
    assert route(4, 4, 4, b_aligned=0)[0] == SIMT            # fewer than eight contiguous elements
    assert route(333, 77, 50, dtype=ek.F32)[0] == F32
    assert route(4096, 4096, 4096, dtype=ek.F32)[0] == F32_WIDE
    assert route(3, 3, 3, dtype=ek.F32)[0] == SIMT
    assert route(3, 3, 3, dtype=ek.F32, residual=1) == ek.ERR_UNSUPPORTED
    assert route(4, 4, 4, dtype=ek.I64) == ek.ERR_UNSUPPORTED
    assert route(4, 4, 0) == route(4, 0, 4) == route(4, 8, 8, lda=4) == ek.ERR_INVALID_ARGUMENT


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
