"""Performance cases of operatorlib: the calls an inference program makes
through ``torch.ops.operatorlib``, over the sizes, data types and options it
makes them with.

``listed()`` holds one representative per operator and regime; ``draw(rng)``
gives further cases of the same ranges. Every case is one operator call on
tensors that are already in device memory, the way a forward pass issues it.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "orin-cuda-operator-library_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import operatorlib  # noqa: E402

operatorlib.load_operatorlib()

EPS = 1e-6
# Floating-point work of the largest listed case; draw() stays under it.
MOST_FLOPS = 4.0 * 4 * 32 * 128 * (8192 * 8193 // 2)
# Elements of the largest row, vector and matrix operand draw() gives.
MOST_ELEMENTS = 1 << 25


def listed():
    return [
        # A large vector summed to one value (statistics over a whole tensor).
        {"name": "reduce_f32", "op": "reduce", "dtype": "f32", "n": 16777216},
        # Scores normalised by rows whose length is no multiple of a vector.
        {"name": "softmax_f32_ragged", "op": "softmax", "dtype": "f32", "rows": 4097, "cols": 1023},
        # The smallest call: the norm of one decode step's hidden states, where
        # launches and latency count.
        {"name": "rmsnorm_f16_decode", "op": "rmsnorm", "dtype": "f16", "rows": 16, "cols": 4096},
        # The norm of a prompt's hidden states.
        {"name": "rmsnorm_f32_prompt", "op": "rmsnorm", "dtype": "f32", "rows": 2048, "cols": 4096},
        # A layout change with both sides off every vector boundary.
        {"name": "transpose_f32_ragged", "op": "transpose", "dtype": "f32", "rows": 4095, "cols": 4097},
        # A projection in a decode step of 16 sequences: a stream over the weights.
        {"name": "gemm_f16_decode", "op": "gemm", "dtype": "f16", "m": 16, "n": 4096, "k": 4096},
        # A projection of a short prompt: too few tokens to fill the GPU with
        # large tiles, too many for a stream.
        {"name": "gemm_f16_short_prompt", "op": "gemm", "dtype": "f16", "m": 300, "n": 4096, "k": 4096},
        # An MLP projection of a long prompt.
        {"name": "gemm_f16_mlp", "op": "gemm", "dtype": "f16", "m": 2000, "n": 11008, "k": 4096},
        # A medium fp32 product.
        {"name": "gemm_f32", "op": "gemm", "dtype": "f32", "m": 1000, "n": 1000, "k": 1000},
        # One sequence's causal attention: few query blocks.
        {"name": "attention_f16_prompt", "op": "attention", "dtype": "f16", "batch": 1, "heads": 12,
         "seq": 1024, "dim": 128, "causal": True},
        # The largest call: a batch of long sequences.
        {"name": "attention_f16_long", "op": "attention", "dtype": "f16", "batch": 4, "heads": 32,
         "seq": 8192, "dim": 128, "causal": True},
        # fp32 attention over an encoder's odd-length sequence, every key visible.
        {"name": "attention_f32_encoder", "op": "attention", "dtype": "f32", "batch": 1, "heads": 12,
         "seq": 1000, "dim": 64, "causal": False},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A feature width: mostly a multiple of 64, now and then any number."""
    w = _log_int(rng, low, high)
    return w if rng.random() < 0.25 else max(low, (w + 32) // 64 * 64)


def draw(rng):
    while True:
        op = rng.choice(["reduce", "softmax", "rmsnorm", "transpose", "gemm", "gemm", "attention", "attention"])
        dtype = "f32" if op in ("reduce", "transpose") or rng.random() < 0.3 else "f16"
        case = {"op": op, "dtype": dtype}
        if op == "reduce":
            case["n"] = _log_int(rng, 4096, MOST_ELEMENTS)
        elif op in ("softmax", "rmsnorm"):
            case["rows"] = _log_int(rng, 1, 8192)
            case["cols"] = _width(rng, 256, 50257 if op == "softmax" else 12288)
            if case["rows"] * case["cols"] > MOST_ELEMENTS:
                continue
        elif op == "transpose":
            case["rows"], case["cols"] = _width(rng, 64, 8192), _width(rng, 64, 8192)
            if case["rows"] * case["cols"] > MOST_ELEMENTS:
                continue
        elif op == "gemm":
            case["m"] = _log_int(rng, 1, 8192)
            case["n"], case["k"] = _width(rng, 512, 12288), _width(rng, 512, 12288)
            if 2.0 * case["m"] * case["n"] * case["k"] > (1.5e11 if dtype == "f32" else 1.1e12):
                continue
        else:
            case["batch"], case["heads"] = _log_int(rng, 1, 8), rng.choice([8, 12, 16, 32])
            case["seq"] = _log_int(rng, 64, 8192)
            case["dim"] = rng.choice([64, 96, 128, 128])
            case["causal"] = rng.random() < 0.6
            if work(case)["flops"] > (2e11 if dtype == "f32" else MOST_FLOPS):
                continue
        return case


def _torch_dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _torch_dtype(case)

    def normal(*shape, scale=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale).to(dt)

    def uniform(*shape, low=-1.0, high=1.0):
        return torch.rand(shape, generator=g, device="cuda").mul_(high - low).add_(low).to(dt)

    op = case["op"]
    if op == "reduce":
        args = (uniform(case["n"]),)
    elif op == "softmax":
        args = (normal(case["rows"], case["cols"], scale=3.0),)
    elif op == "rmsnorm":
        args = (normal(case["rows"], case["cols"]), uniform(case["cols"], low=0.5, high=1.5))
    elif op == "transpose":
        args = (uniform(case["rows"], case["cols"]),)
    elif op == "gemm":
        args = (normal(case["m"], case["k"]),
                normal(case["k"], case["n"], scale=1.0 / math.sqrt(case["k"])))
    else:
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        args = (normal(*shape), normal(*shape), normal(*shape))
    return {"op": op, "args": args, "causal": case.get("causal", False)}


def run(state):
    ops, args = torch.ops.operatorlib, state["args"]
    op = state["op"]
    if op == "reduce":
        return ops.reduce_sum(*args)
    if op == "softmax":
        return ops.softmax(*args)
    if op == "rmsnorm":
        return ops.rmsnorm(*args, EPS)
    if op == "transpose":
        return ops.transpose(*args)
    if op == "gemm":
        return ops.gemm(*args)
    return ops.attention(*args, state["causal"])


def work(case):
    size = 2 if case["dtype"] == "f16" else 4
    op = case["op"]
    if op == "reduce":
        return {"bytes": 4.0 * case["n"] + 4, "flops": 0.0}
    if op == "softmax":
        return {"bytes": 2.0 * size * case["rows"] * case["cols"], "flops": 0.0}
    if op == "rmsnorm":
        return {"bytes": size * (2.0 * case["rows"] * case["cols"] + case["cols"]), "flops": 0.0}
    if op == "transpose":
        return {"bytes": 8.0 * case["rows"] * case["cols"], "flops": 0.0}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": size * (m * k + k * n) + 4.0 * m * n, "flops": 2.0 * m * n * k}
    s, heads = case["seq"], case["batch"] * case["heads"]
    pairs = s * (s + 1) // 2 if case["causal"] else s * s
    return {"bytes": heads * s * case["dim"] * (3.0 * size + 4.0),
            "flops": 4.0 * heads * case["dim"] * pairs}


def tolerance(case):
    """About four times the largest error against 64 bits seen over the ranges:
    5e-7 for fp32 sums (products of up to 12288 terms: 1e-6), 2.1e-4 for fp16
    results, 1.7e-4 for attention on fp16 inputs (its probabilities are
    rounded to fp16). reduce: its terms cancel, so a small sum carries the
    rounding of larger partial sums."""
    op, half = case["op"], case["dtype"] == "f16"
    if op == "transpose":
        return "exact"
    if op == "reduce":
        return {"rel": 1e-5}
    if op in ("softmax", "rmsnorm"):
        return {"rel": 8e-4 if half else 1e-6}
    if op == "gemm":
        return {"rel": 4e-6}
    return {"rel": 8e-4 if half else 2e-6}


def exact(case, seed):
    args = prepare(case, seed)["args"]
    op = case["op"]
    if op == "reduce":
        return args[0].double().sum()
    if op == "softmax":
        return torch.softmax(args[0].double(), dim=-1)
    if op == "rmsnorm":
        x = args[0].double()
        return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * args[1].double()
    if op == "transpose":
        return args[0].double().t().contiguous()
    if op == "gemm":
        return torch.mm(args[0].double(), args[1].double())
    q, k, v = (t.flatten(0, 1) for t in args)
    heads, s, dim = q.shape
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    hidden = torch.ones(s, s, dtype=torch.bool, device=q.device).triu_(1) if case["causal"] else None
    for h in range(heads):
        scores = torch.mm(q[h].double(), k[h].double().t().contiguous()).div_(math.sqrt(dim))
        if hidden is not None:
            scores.masked_fill_(hidden, -math.inf)
        out[h] = torch.mm(torch.softmax(scores, dim=-1), v[h].double())
    return out.view(args[0].shape)
