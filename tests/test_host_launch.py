"""The native half of the launchers: the step loop (on the host), and launches that go by a plan (on the GPU): a plan serves
exactly the calls that agree in layout, alignment and arguments, and gives the first call's bits."""

import contextvars

import pytest
import torch

from helpers import seeded


def _host():
    from torch_mojo_backend import eager_kernels as ek
    return ek.host()


def test_the_step_loop_runs_releases_and_reports():
    node = contextvars.ContextVar("node", default=None)
    seen = []

    def note(*args, **kwargs):
        seen.append((node.get(), args, kwargs))
        return len(seen)

    def fail(x):
        raise ValueError(f"no {x}")

    template = [(note, (None, 7), ((0, 0),), None, (), "a", 1, ()),
                (note, (None, None), ((0, 1), (1, 0)), ("scale",), (2.5,), "b", 2, (1,)),
                (note, (), None, None, (), "c", 3, (0, 2))]
    loop = _host().program(template, lambda i, env: ((i, list(env)), {"late": True}), node)
    env, failed = ["x", None, None, None], []
    assert _host().run(loop, env, failed) is None and failed == []
    assert seen == [("a", ("x", 7), {}), ("b", (1, "x"), {"scale": 2.5}),
                    ("c", (2, ["x", None, 2, None]), {"late": True})]
    assert env == [None, None, None, 3] and node.get() is None
    broken = _host().program([template[0], (fail, (None,), ((0, 1),), None, (), "bad", 2, ())], None, node)
    env = ["x", None, None]
    with pytest.raises(ValueError, match="no 4"):
        _host().run(broken, env, failed)
    assert failed == [1] and env == ["x", 4, None] and node.get() is None
    with pytest.raises(IndexError):
        _host().run(loop, ["x"], failed)


def test_plans_are_for_plain_hip_tensors_only():
    x = torch.zeros(4, 4)
    spec = ("tmb_gelu", 1, (("o", 0), ("t", 0), 16, 0, 0, "stream"), (((4, 4), None, torch.float32),), 0, 0)
    assert _host().keep(spec, 900, 1, x, "none") is False
    assert _host().planned(900, 1, x, "none") is None
    assert _host().planned(900, 1, None, "none") is None and _host().planned(900, 1, x, []) is None
    assert _host().planned("gelu", 1, x) is None


def _calls(ops):
    """name -> (call on fresh tensors of a seed, at an element offset of the first operand)"""
    def first(shape, seed, offset, dtype=torch.bfloat16):
        n = 1
        for d in shape:
            n *= d
        store = torch.empty(n + 8, dtype=dtype, device="cuda")
        return store[offset:offset + n].view(shape).copy_(seeded(shape, seed=seed, dtype=dtype))

    def rest(shape, seed, dtype=torch.bfloat16):
        return seeded(shape, seed=seed + 100, dtype=dtype).cuda()

    heads = lambda seed, offset: first((2, 3, 40, 64), seed, offset)  # noqa: E731
    return {
        "gemm": lambda s, o: ops.gemm(first((33, 64), s, o), rest((48, 64), s).t(), rest((48,), s)),
        "gemm_residual": lambda s, o: ops.gemm(first((33, 64), s, o), rest((48, 64), s).t(), None,
                                               residual=rest((33, 48), s)),
        "bmm": lambda s, o: ops.gemm(first((3, 33, 64), s, o), rest((3, 64, 48), s)),
        "layer_norm": lambda s, o: ops.layer_norm(first((5, 96), s, o), [96], rest((96,), s), None, 1e-5),
        "layer_norm_eps": lambda s, o: ops.layer_norm(first((5, 96), s, o), [96], rest((96,), s), None, 1e-1),
        "softmax": lambda s, o: ops.softmax(first((5, 96), s, o), -1),
        "log_softmax": lambda s, o: ops.softmax(first((5, 96), s, o), -1, log=True),
        "softmax_scaled": lambda s, o: ops.softmax_scaled(first((2, 8, 8), s, o), 0.5, 8),
        "softmax_backward": lambda s, o: ops.softmax_backward(first((5, 96), s, o), rest((5, 96), s), 1, False),
        "sum_rows": lambda s, o: ops.reduce(first((5, 96), s, o), [1], False, 0),
        "sum_keep": lambda s, o: ops.reduce(first((5, 96), s, o), [1], True, 0),
        "sum_cols": lambda s, o: ops.reduce(first((512, 96), s, o), [0], True, 0),
        "argmax": lambda s, o: ops.argmax(first((5, 96), s, o), 1, False),
        "embedding": lambda s, o: ops.embedding(first((50, 96), s, o), torch.arange(7, device="cuda") * (s % 5)),
        "gelu": lambda s, o: ops.gelu(first((5, 96), s, o), "tanh"),
        "gelu_backward": lambda s, o: ops.gelu_backward(first((5, 96), s, o), rest((5, 96), s), "none"),
        "attention": lambda s, o: ops.attention(heads(s, 0), heads(s + 1, 0), heads(s + 2, 0), 0.125, True,
                                                return_lse=True, like_query=True),
        "attention_f32": lambda s, o: ops.attention_f32(*(heads(s + i, 0).float() for i in range(3)), 0.125, False),
        "decode_append": lambda s, o: ops.attention_decode_append(
            heads(s, 0)[:, :, :1], heads(s + 1, 0), heads(s + 2, 0), rest((2, 3, 1, 64), s), rest((2, 3, 1, 64), s + 1),
            0.125),
        "norm_backward": lambda s, o: ops.layer_norm_backward(
            first((5, 96), s, o), rest((5, 96), s), [96], rest((5, 1), s, torch.float32),
            rest((5, 1), s + 1, torch.float32).abs(), rest((96,), s), [True, False, True]),
        "norm_backward_add": lambda s, o: ops.layer_norm_backward_add(
            first((64, 768), s, o), rest((64, 768), s), [768], rest((64, 1), s, torch.float32),
            rest((64, 1), s + 1, torch.float32).abs(), rest((768,), s), rest((64, 768), s + 2), True),
    }


@pytest.mark.gpu
def test_a_planned_launch_gives_the_bits_of_the_first():
    from torch_mojo_backend.eager_kernels import hip_ops as ops

    flat = lambda r: [t for t in (r if isinstance(r, tuple) else (r,))]  # noqa: E731
    for offset in (0, 1):       # on and off a 16-byte boundary
        for name, call in _calls(ops).items():
            wanted = []
            for seed in (1, 2):
                _host().forget()                # no plan: the launcher in Python
                wanted.append(flat(call(seed, offset)))
            hits = []
            real = ops._planned

            def watched(*a, _real=real):
                done = _real(*a)
                hits.append(done is not None)
                return done

            ops._planned = watched
            try:
                for seed in (1, 2, 1):
                    got = flat(call(seed, offset))
                    for g, w in zip(got, wanted[seed - 1], strict=True):
                        assert (g is None) == (w is None), name
                        if w is not None:
                            assert g.shape == w.shape and g.stride() == w.stride() and g.dtype == w.dtype, name
                            assert torch.equal(g, w), (name, offset, seed)
            finally:
                ops._planned = real
            # (a call that the kernels leave to its caller has no plan)
            assert wanted[0] == [None] or (all(hits) and hits), (name, offset)


@pytest.mark.gpu
def test_a_plan_is_not_used_where_layout_or_arguments_differ():
    from torch_mojo_backend.eager_kernels import hip_ops as ops

    x = seeded((6, 96), seed=3).cuda()
    _host().forget()
    assert torch.equal(ops.reduce(x, [1], False, 0), ops.reduce(x, [1], False, 0))
    want = x.double().sum(0).float()
    torch.testing.assert_close(ops.reduce(x, [0], False, 0), want)
    torch.testing.assert_close(ops.reduce(x.t().contiguous().t(), [1], False, 0), x.double().sum(1).float())
    assert ops.reduce(x, [1], True, 0).shape == (6, 1)
    g = torch.ones(96, device="cuda")
    a, b = (ops.layer_norm(x, [96], g, None, eps)[0] for eps in (1e-5, 10.0))
    assert not torch.equal(a, b)
    assert ops.layer_norm(x, [96], g, None, 1e-5, need_stats=False)[1] is None

    # a number in a tensor may have changed since the call that left a plan
    for number in (torch.tensor(1e-5), torch.tensor(1e-5).numpy()):
        for value in (1e-5, 10.0, 1e-5):
            number[...] = value
            got = [ops.layer_norm(x, [96], g, None, number)[0] for _ in range(2)]
            assert torch.equal(got[0], b if value > 1 else a) and torch.equal(got[1], got[0])

    class Wrapped(torch.Tensor):
        pass

    assert _host().planned(ops._OP_REDUCE, 1, x.as_subclass(Wrapped), (1,), False, 0) is None
    with pytest.raises(ValueError):
        ops.layer_norm(x, [95], g, None, 1e-5)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                       # the plan launches on the caller's stream
        out = ops.gelu(ops.gelu(x, "tanh"), "tanh")
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, ops.gelu(ops.gelu(x, "tanh"), "tanh"))


@pytest.mark.gpu
def test_plans_in_use_outlast_the_plans_of_many_layouts():
    """As many layouts as three tables hold: the plan that every few of them use is there throughout, the first ones go."""
    from torch_mojo_backend import eager_kernels as ek

    host, x = _host(), torch.ones(4, 4, device="cuda")
    host.forget()
    spec = ("tmb_gelu", ek.address("tmb_gelu"), (("o", 0), ("t", 0), 16, ek.F32, 0, "stream"),
            (((4, 4), None, torch.float32),), 0, 0)
    assert host.keep(spec, 901, 1, x, "often") is True and host.planned(901, 1, x, "often") is not None
    for i in range(3 * 8192):
        assert host.keep(spec, 900, 1, x, i) is True
        if i % 1000 == 0:
            assert host.planned(901, 1, x, "often") is not None, i
    assert host.planned(900, 1, x, 0) is None and host.planned(900, 1, x, 8192) is None
    assert host.planned(900, 1, x, 3 * 8192 - 1) is not None and host.planned(900, 1, x, 2 * 8192 + 9) is not None
    host.forget()
    assert host.planned(901, 1, x, "often") is None
