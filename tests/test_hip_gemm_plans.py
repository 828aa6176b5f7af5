"""A product with a residual whose layout has been launched before goes straight to the launch: the same bits as the
first call, and only for calls that agree in everything the checks look at."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mnk", [(128, 768, 768), (37, 130, 77), (1332, 768, 3072)])
def test_a_remembered_residual_launch(dtype, mnk):
    from torch_mojo_backend.eager_kernels import hip_ops
    m, n, k = mnk
    g = torch.Generator(device="cuda").manual_seed(m)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)  # noqa: E731
    a, w, bias, r = make(m, k), make(n, k), make(n), make(m, n)
    first = hip_ops.gemm(a, w.t(), bias, residual=r)
    assert torch.equal(hip_ops.gemm(a, w.t(), bias, residual=r), first)
    # other tensors of the same layout, then a residual and an operand of another
    a2, r2 = make(m, k), make(m, n)
    want = a2.double() @ w.double().t().contiguous() + bias.double() + r2.double()
    tol = {torch.bfloat16: 2.0 ** -8, torch.float32: (k + 2) * 2.0 ** -24}[dtype]
    scale = a2.double().abs() @ w.double().abs().t().contiguous() + bias.double().abs() + r2.double().abs()
    slack = tol * want.abs() + (k + 2) * 2.0 ** -24 * scale
    strided = torch.empty(m, n + 3, device="cuda", dtype=dtype)[:, :n].copy_(r2)
    shifted = torch.empty(m * k + 1, device="cuda", dtype=dtype)[1:].view(m, k).copy_(a2)
    for x in (a2, shifted):
        for res in (r2, strided, r2.t().contiguous().t()):
            for _ in range(2):
                assert ((hip_ops.gemm(x, w.t(), bias, residual=res).double() - want).abs() <= slack).all()
    wide = hip_ops.gemm(a2, w.t(), bias, residual=r2.float(), out_dtype=torch.float32)
    assert wide.dtype == torch.float32 and torch.equal(
        hip_ops.gemm(a2, w.t(), bias, residual=r2.float(), out_dtype=torch.float32), wide)
    with pytest.raises(ValueError):
        hip_ops.gemm(a, w.t(), bias, residual=r[:, :-1])
