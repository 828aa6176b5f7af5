"""GPU parity of the float32 fused attention, forward and backward, against float64, inside the
a-priori error bound of float32 sums of these lengths."""

import pytest
import torch

from helpers import seeded

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _ops():
    from torch_mojo_backend.eager_kernels import hip_ops
    return hip_ops


def _reference(q, k, v, dout, scale, causal):
    """float64 results and, per result, how far float32 sums may be off it: a score is a sum of 64 products
    and one more rounding, so a probability is off by twice that relative to itself; a result is a
    sum over the keys (queries) of terms with that error."""
    q, k, v, g = (x.double() for x in (q, k, v, dout.transpose(1, 2)))
    s = q @ k.transpose(-1, -2) * scale
    t, n = s.shape[-2:]
    if causal:
        s = s.masked_fill(torch.ones(t, n, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    out = p @ v
    delta = (g * out).sum(-1, keepdim=True)
    ds = p * (g @ v.transpose(-1, -2) - delta) * scale
    grads = (ds.transpose(-1, -2) @ q, ds @ k, p.transpose(-1, -2) @ g)     # dk, dq, dv
    rel = 2 * 66 * EPS * scale * (q.abs() @ k.abs().transpose(-1, -2)).max().item() + 8 * EPS
    ds_abs = p * (g.abs() @ v.abs().transpose(-1, -2) + (g.abs() * (p @ v.abs())).sum(-1, keepdim=True)) * scale
    off = lambda terms, length: (2 * rel + (length + 140) * EPS) * terms    # noqa: E731
    return (out, grads[1], grads[0], grads[2]), (
        off(p @ v.abs(), n), off(ds_abs @ k.abs(), n), off(ds_abs.transpose(-1, -2) @ q.abs(), t),
        off(p.transpose(-1, -2) @ g.abs(), t))


# around the 32-row block and the four waves that share it, unequal counts, more heads than one chunk of them,
# an odd number of heads over several blocks
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 31, 31), (1, 2, 32, 32), (1, 2, 33, 33), (2, 2, 97, 97),
                                   (1, 3, 128, 128), (2, 2, 129, 129), (5, 13, 65, 65), (1, 2, 77, 150),
                                   (1, 2, 150, 77), (1, 2, 3, 300), (1, 2, 300, 3), (1, 12, 333, 333)])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_f32_matches_float64(shape, causal):
    b, h, t, s = shape
    packed = t == s
    if packed:  # slices of one projection, and gradients into one buffer
        buf = seeded((b, t, 3, h, 64), seed=t)
        (q, k, v), (q_d, k_d, v_d) = (x.permute(2, 0, 3, 1, 4) for x in (buf, buf.cuda()))
    else:
        q, k, v = (seeded((b, h, n, 64), seed=t + i) for i, n in enumerate((t, s, s)))
        q_d, k_d, v_d = q.cuda(), k.cuda(), v.cuda()
    dout = seeded((b, t, h, 64), seed=t + 7)
    ops = _ops()
    out, stats = ops.attention_f32(q_d, k_d, v_d, 0.125, causal, return_stats=True)
    grads = ops.attention_f32_backward(dout.cuda().transpose(1, 2), q_d, k_d, v_d, out.transpose(1, 2), stats, 0.125,
                                       causal, packed=packed)
    want, bounds = _reference(q, k, v, dout, 0.125, causal)
    for name, got, ref, bound in zip(("out", "dq", "dk", "dv"), (out.transpose(1, 2), *grads), want, bounds):
        assert got.shape == ref.shape, name
        worst = ((got.cpu().double() - ref).abs() - bound).max().item()
        assert worst <= 0, (name, worst)
    again = ops.attention_f32(q_d, k_d, v_d, 0.125, causal)
    assert torch.equal(again, out)


def test_attention_f32_with_scores_far_apart_infinite_and_nan():
    q, k, v = (seeded((1, 1, 70, 64), seed=i, scale=8.0) for i in range(3))
    q[0, 0, 5] = 0.0                      # equal scores
    q[0, 0, :, 1] = 1.0
    k[0, 0, 0, 1] = -float("inf")         # all that query 0 sees: 0 / 0, as a softmax has it; nothing to the others
    q[0, 0, 5, 1] = 1.0
    k[0, 0, 40, 3] = float("nan")         # queries 40.. see it
    got = _ops().attention_f32(q.cuda(), k.cuda(), v.cuda(), 0.125, True).transpose(1, 2).cpu()[0, 0]
    s = (q.double() @ k.double().transpose(-1, -2) * 0.125).masked_fill(
        torch.ones(70, 70, dtype=torch.bool).triu(1), float("-inf"))
    want = (torch.softmax(s, -1) @ v.double())[0, 0]
    assert torch.isnan(got[0]).all() and torch.isnan(got[40:]).all()
    # |score| stays below 500: 66 roundings of it in an exponent, on values below 40
    torch.testing.assert_close(got[1:40].double(), want[1:40], rtol=0, atol=2 * 40 * 66 * EPS * 500)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_f32_with_values_that_are_not_finite(bad):
    """Row 70 of one operand, in the third block of 32 of five: what sees it is not finite, what does not and shares no
    block with what does has the bits that it has without."""
    q, k, v, dout = (seeded((1, 2, 150, 64), seed=i).cuda() for i in range(4))
    ops = _ops()

    def run(q, k, v, dout):
        out, stats = ops.attention_f32(q, k, v, 0.125, True, return_stats=True)
        return out.transpose(1, 2), *ops.attention_f32_backward(dout, q, k, v, out.transpose(1, 2), stats, 0.125, True)

    def spoilt(x):
        x = x.clone()
        x[:, :, 70] = bad
        return x

    clean = run(q, k, v, dout)
    out, dq, dk, dv = run(q, k, spoilt(v), dout)
    assert not out[:, :, 70:].isfinite().any() and not dq[:, :, 70:].isfinite().any()
    assert torch.equal(out[:, :, :64], clean[0][:, :, :64]) and torch.equal(dq[:, :, :64], clean[1][:, :, :64])
    _, _, dk, dv = run(q, k, v, spoilt(dout))       # query 70 sees keys 0 .. 70
    assert not dk[:, :, :71].isfinite().any() and not dv[:, :, :71].isfinite().any()
    assert torch.equal(dk[:, :, 96:], clean[2][:, :, 96:]) and torch.equal(dv[:, :, 96:], clean[3][:, :, 96:])


def test_a_float32_graph_runs_one_fused_attention_per_block(monkeypatch):
    from demo_scripts.gpt2 import build_gpt2_small, seeded_tokens
    from torch_mojo_backend import mojo_backend

    ops = _ops()
    calls = []
    real = ops.attention_f32
    monkeypatch.setattr(ops, "attention_f32", lambda *a, **kw: (calls.append(1), real(*a, **kw))[1])
    idx = seeded_tokens(3, 77, seed=1)
    with torch.no_grad():
        want, _ = build_gpt2_small(seed=0, n_layer=2).double()(idx)
        got, _ = torch.compile(build_gpt2_small(seed=0, n_layer=2).cuda(), backend=mojo_backend, fullgraph=True)(idx.cuda())
        assert len(calls) == 2
        blind = build_gpt2_small(seed=0, n_layer=2).cuda()
        for block in blind.transformer.h:
            block.attn.bias[0, 0, 5, 40] = 1.0          # not causal any more: op by op
        torch.compile(blind, backend=mojo_backend, fullgraph=True)(idx.cuda())
    assert len(calls) == 2
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("scale", [0.1, 0.3, 1.0 / 7.0])
def test_the_backward_has_the_probabilities_of_the_forward(scale):
    """One key: its probability is exp(0) / 1, exactly, where the backward rounds the scaled score as the forward did whose
    maximum it takes off. (Scores of 1e6: their rounding is some hundredths.)"""
    q, k, v, dout = (seeded((2, 3, 1, 64), seed=i, scale=200.0 if i < 2 else 1.0).cuda() for i in range(4))
    ops = _ops()
    out, stats = ops.attention_f32(q, k, v, scale, True, return_stats=True)
    _, _, dv = ops.attention_f32_backward(dout, q, k, v, out.transpose(1, 2), stats, scale, True)
    assert torch.equal(out.transpose(1, 2), v) and torch.equal(dv, dout)
