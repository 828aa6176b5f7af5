"""What a program that uses this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values. ``prepare`` makes what the program holds before the call (device
tensors, a compiled model), ``run`` is one pass through the public entry points, ``work`` the bytes
and operations that pass cannot do without, ``tolerance`` how far another correct implementation at
the same precision may be off.

The entry points are the two a process can use side by side: ``torch.compile(..,
backend=mojo_backend)`` for models (forward, training step, decode step) and the aten registry
``MAPPING_TORCH_ATEN_TO_MOJO`` for single ops. The eager ``mojo`` device is left out: a process
that has registered it can no longer differentiate plain HIP tensors, and its ops end in the same
launchers as the registry's.
"""

from __future__ import annotations

import functools
import math
import os
import sys

import torch
import torch.nn.functional as F

_PACKAGE = os.path.join(os.getcwd(), "torch-max-backend_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from demo_scripts.gpt2 import GPT, GPTConfig  # noqa: E402
from torch_mojo_backend import MAPPING_TORCH_ATEN_TO_MOJO, mojo_backend  # noqa: E402

aten = torch.ops.aten

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}
_LAYERS, _HEADS, _WIDTH, _VOCAB, _CONTEXT = 12, 12, 768, 50257, 1024
_BLOCK_WEIGHTS = 12 * _WIDTH * _WIDTH                       # matrices of one decoder block
_WEIGHTS = _LAYERS * _BLOCK_WEIGHTS + (_VOCAB + _CONTEXT) * _WIDTH

# One program compiles its models for many batch sizes and lengths: every shape is its own static
# graph, more of them than dynamo keeps for one function by default.
torch._dynamo.config.recompile_limit = 256
torch._dynamo.config.accumulated_recompile_limit = 1024


def listed():
    return [
        # The workload's small configuration: one short prompt, where the host's step per node and
        # the latency of every launch count.
        {"name": "forward_bf16_1x128", "kind": "forward", "dtype": "bf16", "batch": 1, "seq": 128, "replay": False},
        # A few ragged prompts served through recorded graphs, the option for launch-bound models.
        {"name": "forward_bf16_3x77_replay", "kind": "forward", "dtype": "bf16", "batch": 3, "seq": 77, "replay": True},
        # Evaluation in full precision at an odd length: attention runs unfused there.
        {"name": "forward_fp32_4x333", "kind": "forward", "dtype": "fp32", "batch": 4, "seq": 333, "replay": False},
        # The workload's large configuration: prefill / scoring throughput.
        {"name": "forward_bf16_32x1024", "kind": "forward", "dtype": "bf16", "batch": 32, "seq": 1024, "replay": False},
        # A training step (forward, cross-entropy, backward) at the benchmark's batch.
        {"name": "train_bf16_16x1024", "kind": "train", "dtype": "bf16", "batch": 16, "seq": 1024},
        # The same in full precision on a few short ragged sequences (fine-tuning, gradient checks).
        {"name": "train_fp32_3x250", "kind": "train", "dtype": "fp32", "batch": 3, "seq": 250},
        # One generated token per sequence with a key/value cache, the middle of a generation loop.
        {"name": "decode_bf16_32x499", "kind": "decode", "dtype": "bf16", "batch": 32, "past": 499},
        # The headline product, N-major right operand.
        {"name": "linear_bf16_8192", "kind": "linear", "dtype": "bf16", "m": 8192, "n": 8192, "k": 8192,
         "weight": "kn", "backward": False},
        # A classifier head whose sizes are no multiples of anything, with its backward.
        {"name": "linear_fp16_1999x1001x1500_bwd", "kind": "linear", "dtype": "fp16", "m": 1999, "n": 1001,
         "k": 1500, "weight": "nk", "backward": True},
        # Layer norm and its backward over the activations of the large forward.
        {"name": "norm_bf16_32768x768", "kind": "norm", "dtype": "bf16", "rows": 32768, "cols": 768},
        # Log-softmax and its backward over a vocabulary of odd width.
        {"name": "softmax_bf16_4096x50257_log", "kind": "softmax", "dtype": "bf16", "rows": 4096, "cols": 50257,
         "log": True},
        # Greedy sampling: the next token of every sequence out of its float32 logits.
        {"name": "argmax_fp32_512x50257", "kind": "reduce", "dtype": "fp32", "op": "argmax", "over": "cols",
         "rows": 512, "cols": 50257},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _size(rng, low, high, unit):
    """A size of the range: half of the time a multiple of `unit`, otherwise as it falls."""
    n = _log_int(rng, low, high)
    return max(unit, n // unit * unit) if rng.random() < 0.5 and n >= unit else n


def draw(rng):
    kind = rng.choice(["forward", "forward", "train", "decode", "linear", "linear", "norm", "softmax", "reduce"])
    if kind == "forward":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        most = 4096 if dtype == "fp32" else 32768            # tokens
        seq = _size(rng, 16, _CONTEXT, 64)
        batch = _log_int(rng, 1, max(1, min(32, most // seq)))
        return {"kind": kind, "dtype": dtype, "batch": batch, "seq": seq,
                "replay": batch * seq <= 2048 and rng.random() < 0.5}
    if kind == "train":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        most = 2048 if dtype == "fp32" else 16384
        seq = _size(rng, 64, _CONTEXT, 64)
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 1, max(1, min(16, most // seq))), "seq": seq}
    if kind == "decode":
        return {"kind": kind, "dtype": "bf16", "batch": _log_int(rng, 1, 256), "past": _size(rng, 16, _CONTEXT - 1, 32)}
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        most = 1e11 if dtype == "fp32" else 6e11             # multiply-adds, forward and backward together
        while True:
            case = {"kind": kind, "dtype": dtype, "m": _size(rng, 1, 32768, 64), "n": _size(rng, 64, 50257, 64),
                    "k": _size(rng, 64, 8192, 64), "weight": rng.choice(["nk", "nk", "kn"]),
                    "backward": rng.random() < 0.4}
            if case["backward"]:
                case["weight"] = "nk"                        # linear_backward takes the weight as [n, k]
            if case["m"] * case["n"] * case["k"] * (3 if case["backward"] else 1) <= most:
                return case
    if kind == "norm":
        cols = rng.choice([_WIDTH, 4096, _size(rng, 64, 8192, 8)])
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp32"]), "rows": _log_int(rng, 16, (1 << 27) // cols),
                "cols": cols}
    if kind == "softmax":
        cols = rng.choice([_CONTEXT, 4096, _VOCAB, _size(rng, 64, 16384, 8)])
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp32"]), "rows": _log_int(rng, 16, (1 << 28) // cols),
                "cols": cols, "log": cols == _VOCAB or rng.random() < 0.3}
    op = rng.choice(["sum", "mean", "amax", "argmax"])
    cols = rng.choice([4096, _VOCAB, _size(rng, 64, 16384, 8)])
    return {"kind": "reduce", "dtype": rng.choice(["bf16", "fp32"]), "op": op,
            "over": "cols" if op == "argmax" else rng.choice(["cols", "rows", "all"]),
            "rows": _log_int(rng, 16, (1 << 28) // cols), "cols": cols}


# ---------------------------------------------------------------------------------------------
# The models a program keeps: built and compiled once, fed many batches.
# ---------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _model(dtype):
    """GPT-2 small with the workload's random initialisation."""
    with torch.random.fork_rng(devices=[0]), torch.device("cuda"):
        torch.manual_seed(0)
        model = GPT(GPTConfig())
    return model.to(_DTYPES[dtype]).eval()


@functools.lru_cache(maxsize=None)
def _forward(dtype):
    return torch.compile(_model(dtype), backend=mojo_backend, fullgraph=True, dynamic=False)


@functools.lru_cache(maxsize=None)
def _loss(dtype):
    model = _model(dtype)

    def loss(tokens, targets):
        logits, _ = model(tokens)
        return F.cross_entropy(logits.view(-1, logits.shape[-1]), targets.view(-1))

    return torch.compile(loss, backend=mojo_backend, fullgraph=True, dynamic=False)


@functools.lru_cache(maxsize=None)
def _decode(dtype):
    """One step of a generation loop: the token's keys and values are appended to each layer's
    cache. One graph serves every length (the cache grows by a token per call)."""
    model = _model(dtype)

    def step(token, position, keys, values):
        stem = model.transformer
        batch = token.shape[0]
        x = stem.wte(token) + stem.wpe(position)
        grown_keys, grown_values = [], []
        for block, past_k, past_v in zip(stem.h, keys, values):
            q, k, v = block.attn.c_attn(block.ln_1(x)).split(_WIDTH, dim=2)
            q, k, v = (t.view(batch, 1, _HEADS, _WIDTH // _HEADS).transpose(1, 2) for t in (q, k, v))
            k, v = torch.cat([past_k, k], dim=2), torch.cat([past_v, v], dim=2)
            y = F.scaled_dot_product_attention(q, k, v)
            x = x + block.attn.c_proj(y.transpose(1, 2).reshape(batch, 1, _WIDTH))
            x = x + block.mlp(block.ln_2(x))
            grown_keys.append(k)
            grown_values.append(v)
        logits = model.lm_head(stem.ln_f(x))[:, -1, :]
        return logits, torch.argmax(logits, dim=-1), grown_keys, grown_values

    return torch.compile(step, backend=mojo_backend, fullgraph=True, dynamic=True)


def _normal(gen, *shape, scale=1.0, shift=0.0):
    return torch.randn(shape, generator=gen, device="cuda") * scale + shift


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    if kind in ("forward", "train"):
        shape = (case["batch"], case["seq"])
        state["tokens"] = torch.randint(0, _VOCAB, shape, generator=gen, device="cuda")
        if kind == "forward":
            state["fn"] = _forward(case["dtype"])
        else:
            state["targets"] = torch.randint(0, _VOCAB, shape, generator=gen, device="cuda")
            state["fn"], state["model"] = _loss(case["dtype"]), _model(case["dtype"])
    elif kind == "decode":
        shape = (case["batch"], _HEADS, case["past"], _WIDTH // _HEADS)
        state["fn"] = _decode(case["dtype"])
        state["token"] = torch.randint(0, _VOCAB, (case["batch"], 1), generator=gen, device="cuda")
        state["position"] = torch.full((1,), case["past"], device="cuda")
        for name in ("keys", "values"):
            state[name] = [_normal(gen, *shape, scale=0.5).to(dtype) for _ in range(_LAYERS)]
    elif kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        state["x"] = _normal(gen, m, k).to(dtype)
        state["weight"] = _normal(gen, *((n, k) if case["weight"] == "nk" else (k, n))).to(dtype)
        state["bias"] = _normal(gen, n).to(dtype)
        if case["backward"]:
            state["grad"] = _normal(gen, m, n).to(dtype)
    elif kind == "norm":
        rows, cols = case["rows"], case["cols"]
        state["x"], state["grad"] = _normal(gen, rows, cols, scale=4.0).to(dtype), _normal(gen, rows, cols).to(dtype)
        state["gamma"] = _normal(gen, cols, scale=0.1, shift=1.0).to(dtype)
        state["beta"] = _normal(gen, cols, scale=0.1).to(dtype)
    elif kind == "softmax":
        state["x"] = _normal(gen, case["rows"], case["cols"], scale=4.0).to(dtype)
        state["grad"] = _normal(gen, case["rows"], case["cols"]).to(dtype)
    else:
        # (a mean of their own, so that the sum of all of them is no cancellation)
        state["x"] = _normal(gen, case["rows"], case["cols"], shift=0.5).to(dtype)
        if case["op"] == "argmax" and case["rows"] >= 100:   # ties in one row of a hundred
            tied = state["x"][::100]
            tied[:, case["cols"] // 2] = tied.amax(dim=1)
    return state


def run(state):
    case, op = state["case"], MAPPING_TORCH_ATEN_TO_MOJO
    kind = case["kind"]
    if kind == "forward":
        # the switch is an environment variable that is looked at on each call
        os.environ["TORCH_MOJO_BACKEND_HIP_GRAPH"] = "1" if case["replay"] else "0"
        with torch.no_grad():
            return state["fn"](state["tokens"])[0]
    if kind == "train":
        model = state["model"]
        model.zero_grad(set_to_none=True)
        loss = state["fn"](state["tokens"], state["targets"])
        loss.backward()
        # the gradients in the groups an optimizer has them in: the two tables, then the blocks'
        # matrices (with weight decay) and all vectors (without) as one flat bucket each
        blocks = [p.grad for p in model.transformer.h.parameters() if p.dim() == 2]
        vectors = [p.grad for p in model.parameters() if p.dim() == 1]
        return (loss.detach(), model.transformer.wte.weight.grad, model.transformer.wpe.weight.grad,
                torch.cat([g.view(-1) for g in blocks]), torch.cat(vectors))
    if kind == "decode":
        os.environ["TORCH_MOJO_BACKEND_HIP_GRAPH"] = "0"
        with torch.no_grad():
            logits, _, keys, values = state["fn"](state["token"], state["position"], state["keys"], state["values"])
        return logits, keys, values
    if kind == "linear":
        weight = state["weight"].t() if case["weight"] == "nk" else state["weight"]
        out = op[aten.addmm](state["bias"], state["x"], weight)
        if not case["backward"]:
            return out
        return out, *op[aten.linear_backward](state["x"], state["grad"], state["weight"], (True, True, True))
    if kind == "norm":
        shape = [case["cols"]]
        out, mean, rstd = op[aten.native_layer_norm](state["x"], shape, state["gamma"], state["beta"], 1e-5)
        return out, *op[aten.native_layer_norm_backward](state["grad"], state["x"], shape, mean, rstd,
                                                         state["gamma"], state["beta"], [True, True, True])
    if kind == "softmax":
        name = ("_log_softmax", "_log_softmax_backward_data") if case["log"] else ("_softmax", "_softmax_backward_data")
        out = op[getattr(aten, name[0])](state["x"], -1, False)
        return out, op[getattr(aten, name[1])](state["grad"], out, -1, state["x"].dtype)
    if case["op"] == "argmax":
        return op[aten.argmax](state["x"], -1)
    dims = {"cols": [1], "rows": [0], "all": [0, 1]}[case["over"]]
    return op[getattr(aten, case["op"])](state["x"], dims)


def work(case):
    """Every input read once, every output written once; of attention's products only the half
    that the causal rule leaves."""
    kind, es = case["kind"], _BYTES[case["dtype"]]
    if kind in ("forward", "train"):
        b, t = case["batch"], case["seq"]
        flops = 2 * b * t * (_LAYERS * _BLOCK_WEIGHTS + _VOCAB * _WIDTH) + _LAYERS * 2 * b * t * t * _WIDTH
        if kind == "forward":
            return {"bytes": _WEIGHTS * es + b * t * (8 + _VOCAB * es), "flops": flops}
        return {"bytes": 2 * _WEIGHTS * es + 16 * b * t, "flops": 3 * flops}
    if kind == "decode":
        b, s = case["batch"], case["past"]
        cache = 2 * _LAYERS * b * _WIDTH * es
        return {"bytes": (_WEIGHTS - _CONTEXT * _WIDTH) * es + cache * (2 * s + 1) + b * _VOCAB * es,
                "flops": 2 * b * (_LAYERS * _BLOCK_WEIGHTS + _VOCAB * _WIDTH) + _LAYERS * 4 * b * (s + 1) * _WIDTH}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        operands = m * k + n * k + n
        if not case["backward"]:
            return {"bytes": (operands + m * n) * es, "flops": 2 * m * n * k}
        return {"bytes": (2 * operands + 2 * m * n) * es, "flops": 6 * m * n * k}
    rows, cols = case["rows"], case["cols"]
    if kind == "norm":     # x, dy in; y, dx out; gamma, beta in, their gradients out; mean and rstd out
        return {"bytes": (4 * rows * cols + 4 * cols) * es + 8 * rows, "flops": 16 * rows * cols}
    if kind == "softmax":  # x, grad in; y, grad_in out
        return {"bytes": 4 * rows * cols * es, "flops": 10 * rows * cols}
    results = {"cols": rows, "rows": cols, "all": 1}[case["over"]]
    return {"bytes": rows * cols * es + results * (8 if case["op"] == "argmax" else es), "flops": rows * cols}


# (rel, max) measured against the same path in float64 (float32 for the bf16 models) over the listed
# and some hundred drawn cases, times four; a bf16 training step, whose gradients are off by 1.2e-2
# and whose table gradient adds two parts that nearly cancel, at the most that is useful.
_MEASURED = {
    "forward": {"bf16": (0.023, 0.15), "fp32": (7e-6, 5e-5)},
    "train": {"bf16": (0.03, 0.95), "fp32": (1.2e-5, 2e-3)},
    "decode": {"bf16": (0.025, 0.15)},
    "linear": {"bf16": (0.007, 0.016), "fp16": (9e-4, 2e-3), "fp32": (6e-6, 2e-5)},
    "norm": {"bf16": (0.007, 0.016), "fp32": (1e-6, 5e-6)},
    "softmax": {"bf16": (0.01, 0.5), "fp32": (1e-6, 1e-4)},
    "reduce": {"bf16": (0.007, 0.016), "fp32": (1e-6, 5e-6)},
}


def tolerance(case):
    if case["kind"] == "reduce" and case["op"] in ("amax", "argmax"):
        return "exact"
    rel, largest = _MEASURED[case["kind"]][case["dtype"]]
    return {"rel": rel, "max": largest}
