"""Which kernel the fused attention ops of a compiled graph run on and how their result is laid out: on
the host with a library that only records its launches, and compiled on the GPU."""

import operator
import types

import pytest
import torch


class RecordingLibrary:
    """Answers sizes and routes like the library; launches are noted and succeed."""

    def __init__(self, real):
        self.real, self.launched = real, []

    def __getattr__(self, name):
        if name.endswith(("_bytes", "_pays", "_route")):
            return getattr(self.real, name)
        return lambda *args: (self.launched.append((name, args)), 0)[1]


@pytest.fixture()
def recorded(monkeypatch):
    """Launchers on host tensors, which count as device tensors here."""
    from torch_mojo_backend import aten_functions
    from torch_mojo_backend import eager_kernels as ek
    from torch_mojo_backend.eager_kernels import hip_ops

    lib = RecordingLibrary(ek.lib())
    monkeypatch.setattr(ek, "lib", lambda: lib)
    monkeypatch.setattr(hip_ops, "_stream", lambda: 0)
    monkeypatch.setattr(hip_ops, "require_hip", lambda *a: None)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    node = types.SimpleNamespace(users=[types.SimpleNamespace(target=operator.getitem, args=(None, 0))])
    token = aten_functions.CURRENT_FX_NODE.set(node)
    yield lib
    aten_functions.CURRENT_FX_NODE.reset(token)


def _queries(b, h, t, d, layout):
    if layout == "contiguous":
        return torch.zeros(b, h, t, d, dtype=torch.bfloat16)
    if layout == "token-major":
        return torch.zeros(b, t, h, d, dtype=torch.bfloat16).transpose(1, 2)
    if layout == "head-outermost":
        return torch.zeros(h, b, t, d, dtype=torch.bfloat16).transpose(0, 1)
    return torch.zeros(b, t, 3, h, d, dtype=torch.bfloat16)[:, :, 0].transpose(1, 2)    # out of a packed projection


LAYOUTS = ["contiguous", "token-major", "head-outermost", "packed"]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("t", [1, 2, 5, 16, 17])
@pytest.mark.parametrize("d", [64, 128])
def test_the_flash_result_is_laid_out_like_the_query(recorded, layout, t, d):
    """Views that are legal for the layout the graph was traced with stay legal."""
    from torch_mojo_backend.aten_functions import aten__scaled_dot_product_flash_attention as flash
    if d == 128 and t == 17:
        pytest.skip("PyTorch's own op")
    q = _queries(2, 3, t, d, layout)
    k = v = torch.zeros(2, 3, 300, d, dtype=torch.bfloat16)
    out = flash(q, k, v)[0]
    assert len(recorded.launched) == 1
    assert out.shape == q.shape and out.stride() == torch.empty_like(q).stride()


@pytest.mark.parametrize("layout", LAYOUTS)
def test_the_appending_step_lays_its_result_out_like_the_query(recorded, layout):
    from torch_mojo_backend.eager_kernels import hip_ops
    q, past, new = _queries(2, 3, 1, 64, layout), torch.zeros(2, 3, 9, 64).bfloat16(), torch.zeros(2, 3, 1, 64).bfloat16()
    out, _, _ = hip_ops.attention_decode_append(q, past, past, new, new, 0.125)
    assert out.stride() == torch.empty_like(q).stride()


@pytest.mark.gpu
@pytest.mark.parametrize("t", [2, 5, 16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("token_major", [False, True])
def test_compiled_attention_of_a_few_queries_is_viewed_and_multiplied(t, head_dim, token_major):
    import torch.nn.functional as F
    from torch_mojo_backend import mojo_backend

    def step(q, k, v, w):
        y = F.scaled_dot_product_attention(q, k, v)
        return y @ w, y.reshape(6, t, head_dim) * 2.0, y.transpose(1, 2).reshape(2, t, 3 * head_dim)

    g = torch.Generator(device="cuda").manual_seed(t)

    def rand(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()

    q = rand(2, t, 3, head_dim).transpose(1, 2) if token_major else rand(2, 3, t, head_dim)
    k, v, w = rand(2, 3, 300, head_dim), rand(2, 3, 300, head_dim), rand(head_dim, 32)
    with torch.no_grad():
        got = torch.compile(step, backend=mojo_backend, fullgraph=True)(q, k, v, w)
    scores = q.double() @ k.double().transpose(-1, -2).contiguous() / head_dim ** 0.5
    y = (torch.softmax(scores, -1) @ v.double())
    for x, want in zip(got, (y @ w.double(), y.reshape(6, t, head_dim) * 2.0,
                             y.transpose(1, 2).reshape(2, t, 3 * head_dim))):
        # P is rounded to bf16 in one of the kernels, y once, and the product sums head_dim of them
        assert (x.double() - want).abs().max().item() <= 2.0 ** -7 * (1 + want.abs().max().item())


def _took(recorded):
    return [name for name, _ in recorded.launched]


@pytest.mark.parametrize("scale", [float("nan"), float("inf"), 0.0, -1.0])
def test_scales_the_kernels_do_not_take_go_to_pytorchs_op(recorded, monkeypatch, scale):
    from torch_mojo_backend import aten_functions
    theirs = []
    flash = aten_functions.aten__scaled_dot_product_flash_attention
    monkeypatch.setattr(aten_functions, "aten", types.SimpleNamespace(
        _scaled_dot_product_flash_attention=lambda *a, **k: (theirs.append(1), (None,) * 9)[1]))
    q = torch.zeros(1, 2, 1, 128).bfloat16()
    flash(q, q, q, scale=scale)
    assert theirs == [1] and _took(recorded) == []


@pytest.mark.parametrize("scale", [float("nan"), float("inf"), 0.0, -1.0, 0.5])
def test_only_an_ordinary_scale_makes_a_step_that_appends(scale):
    from torch_mojo_backend.torch_compile_backend.compiler import _GraphFactory
    aten = torch.ops.aten
    graph = torch.fx.Graph()

    def value(node, tokens):
        node.meta["val"] = torch.zeros(1, 2, tokens, 64, dtype=torch.bfloat16)
        return node

    q, past, new = (value(graph.placeholder(name), n) for name, n in (("q", 1), ("past", 8), ("new", 1)))
    k, v = (value(graph.call_function(aten.cat.default, ([past, new], 2)), 9) for _ in range(2))
    flash = graph.call_function(aten._scaled_dot_product_flash_attention.default, (q, k, v), {"scale": scale})
    graph.output((graph.call_function(operator.getitem, (flash, 0)), k, v))
    assert (flash in _GraphFactory._fuse_decode_append(graph)) == (scale == 0.5)


@pytest.mark.parametrize("case,decode", [
    # (batch, heads, queries, keys, head size): one query, whatever the rest
    ((1, 12, 1, 64, 64), True), ((64, 16, 1, 4096, 64), True), ((64, 16, 1, 1024, 128), True),
    # a few queries on few rows, from the keys on where the prefill kernel's serial walk is longer
    ((1, 12, 2, 256, 64), True), ((1, 12, 16, 4096, 64), True), ((4, 12, 4, 1024, 64), True), ((1, 256, 1, 256, 64), True),
    ((1, 12, 2, 255, 64), False), ((4, 12, 4, 64, 128), True),
    # more rows: K and V once per row against once per 128 queries
    ((32, 12, 16, 1024, 64), False), ((32, 12, 2, 1024, 64), False), ((4, 12, 8, 1024, 64), False),
    ((8, 12, 4, 512, 128), False), ((1, 257, 2, 4096, 64), False), ((1, 128, 2, 4096, 64), True)])
def test_a_few_queries_take_the_decode_kernel_where_it_is_the_faster_one(recorded, monkeypatch, case, decode):
    from torch_mojo_backend import aten_functions
    theirs = []
    flash = aten_functions.aten__scaled_dot_product_flash_attention
    monkeypatch.setattr(aten_functions, "aten", types.SimpleNamespace(
        _scaled_dot_product_flash_attention=lambda *a, **k: (theirs.append(1), (None,) * 9)[1]))
    b, h, t, s, d = case
    q = torch.zeros(d, dtype=torch.bfloat16).as_strided((b, h, t, d), (0, 0, 0, 1))    # (only sizes are looked at)
    k = torch.zeros(d, dtype=torch.bfloat16).as_strided((b, h, s, d), (0, 0, 0, 1))
    flash(q, k, k)
    if decode:
        assert _took(recorded) == ["tmb_attention_decode"] and not theirs
    elif d == 64:
        assert _took(recorded) == ["tmb_attention_fwd"] and not theirs
    else:
        assert theirs == [1] and _took(recorded) == []


@pytest.mark.parametrize("devices", [("cuda:0", "cuda:1", "cuda:0"), ("cuda:0", "cuda:0", "cuda:1"),
                                     ("cuda:1", "cuda:0", "cuda:0")])
@pytest.mark.parametrize("checked", [False, True])
def test_attention_refuses_operands_on_two_devices(devices, checked):
    """Also where the caller has checked their layout (`attention_supported` looks at each operand by itself): a launch
    would read another device's memory."""
    from torch_mojo_backend.eager_kernels import hip_ops

    q, k, v = (types.SimpleNamespace(device=torch.device(d)) for d in devices)
    with pytest.raises(TypeError, match="different devices"):
        hip_ops.attention(q, k, v, 0.125, True, checked=checked)
