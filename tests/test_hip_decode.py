"""Decode attention on the GPU: every number of waves per row the kernel runs with, the pass that
appends to the cache while it attends, and the graph rewrite that uses it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _exact(q, k, v, scale, causal=False):
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * scale
    if causal:
        keep = torch.ones(q.shape[2], k.shape[2], dtype=torch.bool, device="cuda").tril()
        s = s.masked_fill(~keep, float("-inf"))
    return torch.softmax(s, -1) @ v.double()


# (batch, heads, queries, keys): one wave per row (few keys, many rows), four, sixteen; key counts around
# a wave's 32 (16 at head size 128) and the waves' shares; keys of one and two steps (8, 4 keys each)
CASES = [(1, 12, 1, 1), (3, 5, 1, 4), (200, 12, 1, 5), (200, 12, 2, 8), (100, 12, 3, 9), (1, 12, 4, 16), (200, 12, 1, 17),
         (1, 12, 1, 31), (1, 12, 1, 33), (1, 12, 1, 300), (2, 12, 3, 1025), (64, 12, 1, 129), (200, 12, 1, 65),
         (1, 2, 16, 257), (43, 12, 4, 40)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype,head_dim", [(torch.bfloat16, 64), (torch.float16, 128)])
@pytest.mark.parametrize("causal", [False, True])
def test_decode_rows_shared_by_waves(case, dtype, head_dim, causal):
    from torch_mojo_backend.eager_kernels import hip_ops
    b, h, t, s = case
    g = torch.Generator(device="cuda").manual_seed(s)
    q, k, v = (_rand(g, b, h, n, head_dim, dtype=dtype) for n in (t, s, s))
    want = _exact(q, k, v, 0.125, causal)
    for token_major in (False, True):
        got = hip_ops.attention_decode(q, k, v, 0.125, causal, token_major=token_major)
        # float32 inside, one rounding of values up to max|v|
        ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        assert ((got.double() - want).abs() <= ulp * want.abs() + 1e-4).all()


@pytest.mark.parametrize("case", [(1, 12, 1), (3, 12, 6), (200, 12, 7), (200, 12, 15), (200, 12, 16), (3, 12, 32), (32, 12, 499), (180, 12, 70), (2, 3, 2000)])
@pytest.mark.parametrize("dtype,head_dim", [(torch.bfloat16, 64), (torch.float16, 128)])
def test_append_and_attend_in_one_pass(case, dtype, head_dim):
    from torch_mojo_backend.eager_kernels import hip_ops
    b, h, past = case
    g = torch.Generator(device="cuda").manual_seed(past)
    packed = _rand(g, b, 1, 3 * h * head_dim, dtype=dtype)     # q, k, v of the new token as they come
    q, kn, vn = (x.view(b, 1, h, head_dim).transpose(1, 2) for x in packed.split(h * head_dim, dim=2))
    kp, vp = _rand(g, b, h, past, head_dim, dtype=dtype), _rand(g, b, h, past, head_dim, dtype=dtype)
    out, k, v = hip_ops.attention_decode_append(q, kp, vp, kn, vn, 0.125)
    assert torch.equal(k, torch.cat([kp, kn], 2)) and torch.equal(v, torch.cat([vp, vn], 2))
    assert torch.equal(out, hip_ops.attention_decode(q, k, v, 0.125, False))
    assert hip_ops.attention_decode_append(q.float(), kp.float(), vp.float(), kn.float(), vn.float(), 0.125) is None


@pytest.mark.parametrize("keys", [40, 300])
def test_scores_of_minus_infinity_weigh_nothing(keys):
    """Every first key of a wave's share scores -inf: the others decide, as in ATen."""
    from torch_mojo_backend.eager_kernels import hip_ops
    g = torch.Generator(device="cuda").manual_seed(keys)
    q, k, v = (_rand(g, 1, 2, n, 64, dtype=torch.bfloat16) for n in (1, keys, keys))
    q[..., 0] = 1.0
    k[:, :, :keys // 2, 0] = -float("inf")
    want = _exact(q, k, v, 0.125)
    got = hip_ops.attention_decode(q, k, v, 0.125, False)
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("dynamic", [False, True])
def test_a_compiled_decode_step_appends_while_it_attends(dynamic):
    import torch.nn.functional as F
    from torch_mojo_backend import mojo_backend
    from torch_mojo_backend.eager_kernels import hip_ops

    def step(x, w, kp, vp):
        b = x.shape[0]
        q, kn, vn = (y.view(b, 1, 2, 64).transpose(1, 2) for y in (x @ w).split(128, dim=2))
        k, v = torch.cat([kp, kn], 2), torch.cat([vp, vn], 2)
        y = F.scaled_dot_product_attention(q, k, v)
        return y.transpose(1, 2).reshape(b, 1, 128), k, v

    calls = []
    real = hip_ops.attention_decode_append
    hip_ops.attention_decode_append = lambda *a: (calls.append(1), real(*a))[1]
    try:
        torch._dynamo.reset()
        fn = torch.compile(step, backend=mojo_backend, fullgraph=True, dynamic=dynamic)
        g = torch.Generator(device="cuda").manual_seed(3)
        x, w = _rand(g, 3, 1, 128), _rand(g, 128, 384) * 0.1
        kp, vp = _rand(g, 3, 2, 40, 64), _rand(g, 3, 2, 40, 64)
        with torch.no_grad():
            for _ in range(4):     # the cache grows by a token per step
                y, k, v = fn(x, w, kp, vp)
                q = (x @ w)[..., :128].view(3, 1, 2, 64).transpose(1, 2)
                assert torch.equal(k[:, :, :-1], kp) and torch.equal(v[:, :, :-1], vp)
                want = _exact(q, k, v, 0.125).transpose(1, 2).reshape(3, 1, 128)
                # (the query was rounded by another product: a unit of it moves the result)
                assert (y.double() - want).abs().max().item() <= 5e-2
                kp, vp = k, v
    finally:
        hip_ops.attention_decode_append = real
    assert len(calls) >= 1
    torch._dynamo.reset()
