"""The work a program built on this framework has it do, as cases that can be timed and compared.

Each case goes through a public entry point: a torch module compiled for the rocm target and called on device tensors, a
function under ``@native(target="rocm")`` called on numpy arrays, or one of the library-node launchers of
``docc_amd.runtime`` on device memory. ``listed()`` holds one case of each use, ``draw`` more of the same ranges; ``prepare``
makes what the program has in hand before a call, ``run`` is one call, ``work`` what the call cannot do without.

Programs are compiled once per shape and take their weights as arguments, as a program that serves many batches keeps them.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import scipy.special
import torch
import torch.nn.functional as F

from docc_amd import runtime as rt
from docc_amd.python import native
from docc_amd.torch import compile_torch

_TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
_BYTES = {"f64": 8, "f32": 4, "bf16": 2}
#: dense matrix rates (FLOP/s) and the memory rate (bytes/s) by which a drawn case's cost is bounded
_RATE = {"f64": 78.6e12, "f32": 157.3e12, "bf16": 2516.6e12}
_MEMORY_RATE = 8.0e12
_MOST_SECONDS = 1.0e-4


def listed():
    return [
        # a transformer's feed-forward block on a small batch: a few microseconds a kernel, launches count
        {"name": "mlp_f32_1024tok", "op": "mlp", "dtype": "f32", "tokens": 1024, "width": 256},
        # the same block over a prompt in bf16: two large products with elementwise work and a normalisation around them
        {"name": "mlp_bf16_4096tok", "op": "mlp", "dtype": "bf16", "tokens": 4096, "width": 2048},
        # the same block while tokens are generated: a few rows against the whole weights
        {"name": "mlp_bf16_8tok", "op": "mlp", "dtype": "bf16", "tokens": 8, "width": 2048},
        # causal attention over a prompt
        {"name": "attention_prefill", "op": "attention", "batch": 8, "heads": 16, "sq": 2048, "skv": 2048, "dim": 64, "causal": True},
        # one new query per sequence against the keys and values so far
        {"name": "attention_decode", "op": "attention", "batch": 16, "heads": 16, "sq": 1, "skv": 4096, "dim": 128, "causal": False},
        # an encoder's attention at a length of no whole tiles
        {"name": "attention_333", "op": "attention", "batch": 16, "heads": 12, "sq": 333, "skv": 333, "dim": 64, "causal": False},
        # a residual block of a convolutional network on large images
        {"name": "conv_block_56", "op": "conv", "batch": 32, "channels": 64, "out": 64, "size": 56, "stride": 1},
        # the block between two stages: strides of two, a 1x1 projection beside it
        {"name": "conv_block_28s2", "op": "conv", "batch": 32, "channels": 128, "out": 256, "size": 28, "stride": 2},
        # the softmax node over the last axis of a large tensor
        {"name": "softmax_8192x4096", "op": "softmax", "dtype": "f32", "outer": 8192, "reduce": 4096, "inner": 1},
        # the GEMM node in double precision, the size of numpy programs
        {"name": "gemm_f64_1000", "op": "gemm", "dtype": "f64", "m": 1000, "n": 1000, "k": 1000, "trans_b": False},
        # the GEMM node in bf16, large
        {"name": "gemm_bf16_4096", "op": "gemm", "dtype": "bf16", "m": 4096, "n": 4096, "k": 4096, "trans_b": False},
        # a numpy program: host arrays in, a host array out
        {"name": "native_softmax", "op": "native", "outer": 32 * 8 * 256, "reduce": 256},
    ]


def _between(rng, low, high):
    """A whole number of [low, high], spread over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _size(rng, low, high, step):
    """A size of [low, high]: half of them multiples of `step`, the others as they come."""
    v = _between(rng, low, high)
    return v if rng.random() < 0.5 else max(step, v // step * step)


def _draw_once(rng):
    op = rng.choice(["mlp", "mlp", "attention", "attention", "conv", "softmax", "gemm", "gemm", "native"])
    if op == "mlp":
        # from one generated token to a batch of prompts; widths are those of layers: multiples of 64, now and then of 8
        return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "tokens": _size(rng, 1, 8192, 64),
                "width": _between(rng, 16, 384) * 8 if rng.random() < 0.25 else _between(rng, 2, 48) * 64}
    if op == "attention":
        c = {"op": op, "batch": _between(rng, 1, 32), "heads": rng.choice([4, 8, 12, 16, 32]), "dim": rng.choice([32, 64, 64, 128, 128])}
        if rng.random() < 0.4:      # tokens are generated: one query, or the few of a speculated run
            return {**c, "sq": rng.choice([1, 1, 1, 4]), "skv": _size(rng, 32, 32768, 64), "causal": False}
        s = _size(rng, 16, 4096, 64)
        return {**c, "sq": s, "skv": s, "causal": rng.random() < 0.5}
    if op == "conv":
        stride = rng.choice([1, 1, 2])
        channels = _between(rng, 2, 32) * 16
        return {"op": op, "batch": _between(rng, 1, 64), "channels": channels, "out": channels * stride, "size": rng.randint(7, 64), "stride": stride}
    if op == "softmax":
        dtype = rng.choice(["f32", "f32", "f64"])
        return {"op": op, "dtype": dtype, "outer": _between(rng, 1, 65536), "reduce": _size(rng, 16, 65536, 64),
                "inner": 1 if rng.random() < 0.7 else _size(rng, 2, 2048, 16)}
    if op == "gemm":
        return {"op": op, "dtype": rng.choice(["f64", "f32", "bf16"]), "m": _size(rng, 1, 8192, 64), "n": _size(rng, 32, 8192, 64),
                "k": _size(rng, 32, 8192, 64), "trans_b": rng.random() < 0.5}
    return {"op": op, "outer": _between(rng, 16, 65536), "reduce": _size(rng, 16, 4096, 64)}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / _MEMORY_RATE, w["flops"] / _RATE["f32" if case["op"] == "conv" else case.get("dtype", "bf16")])


def draw(rng):
    """One more case of the ranges above: from calls that only launches take time of to the largest listed."""
    while True:
        case = _draw_once(rng)
        if _cost(case) > _MOST_SECONDS or (case["op"] == "native" and work(case)["bytes"] > 2 * 4 * 32 * 8 * 256 * 256):
            continue
        if any(all(c[k] == v for k, v in case.items()) for c in listed() if c["op"] == case["op"]):
            continue
        return case


class _Mlp(torch.nn.Module):
    """LayerNorm, Linear, GELU, Linear and the residual around them."""

    def __init__(self, width):
        super().__init__()
        self.width = width

    def forward(self, x, norm_w, norm_b, w1, b1, w2, b2):
        h = F.layer_norm(x, (self.width,), norm_w, norm_b)
        return x + F.linear(F.gelu(F.linear(h, w1, b1)), w2, b2)


class _ConvBlock(torch.nn.Module):
    """Two 3x3 convolutions (their normalisations folded into weights and bias) and the residual around them; where the
    block halves the image the residual is projected by a 1x1 convolution."""

    def __init__(self, stride, projected):
        super().__init__()
        self.stride, self.projected = stride, projected

    def forward(self, x, w1, b1, w2, b2, w3, b3):
        y = torch.relu(F.conv2d(x, w1, b1, stride=self.stride, padding=1))
        y = F.conv2d(y, w2, b2, padding=1)
        if self.projected:
            x = F.conv2d(x, w3, b3, stride=self.stride)
        return torch.relu(y + x)


@functools.lru_cache(maxsize=None)
def _program(module, arguments, *sizes):
    """`module(*arguments)` compiled for the rocm target, one program per set of `sizes` and kept: it compiles on its first call."""
    return compile_torch(module(*arguments), None, target="rocm")


@native(target="rocm")
def _softmax_rows(x):
    return scipy.special.softmax(x, axis=-1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]

    def normal(*shape, dtype=torch.float32, scale=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * scale).to(dtype)

    if op == "mlp":
        dtype, w = _TORCH[case["dtype"]], case["width"]
        args = (normal(case["tokens"], w, dtype=dtype), 1 + normal(w, dtype=dtype, scale=0.1), normal(w, dtype=dtype, scale=0.1),
                normal(4 * w, w, dtype=dtype, scale=w ** -0.5), normal(4 * w, dtype=dtype, scale=0.1),
                normal(w, 4 * w, dtype=dtype, scale=(4 * w) ** -0.5), normal(w, dtype=dtype, scale=0.1))
        return {"case": case, "program": _program(_Mlp, (w,), case["dtype"], case["tokens"]), "args": args}
    if op == "conv":
        c, o = case["channels"], case["out"]
        projected = case["stride"] != 1 or c != o
        args = (normal(case["batch"], c, case["size"], case["size"]),
                normal(o, c, 3, 3, scale=(2.0 / (9 * c)) ** 0.5), normal(o, scale=0.1),
                normal(o, o, 3, 3, scale=(2.0 / (9 * o)) ** 0.5), normal(o, scale=0.1),
                normal(o, c, 1, 1, scale=(2.0 / c) ** 0.5), normal(o, scale=0.1))
        return {"case": case, "program": _program(_ConvBlock, (case["stride"], projected), case["batch"], c, o, case["size"]), "args": args}
    if op == "attention":
        B, H, D = case["batch"], case["heads"], case["dim"]
        q = normal(B, H, case["sq"], D, dtype=torch.bfloat16)
        k, v = (normal(B, H, case["skv"], D, dtype=torch.bfloat16) for _ in range(2))
        return {"case": case, "q": q, "k": k, "v": v, "o": torch.empty_like(q)}
    if op == "softmax":
        x = normal(case["outer"], case["reduce"], case["inner"], dtype=_TORCH[case["dtype"]], scale=8.0)
        return {"case": case, "x": x, "y": torch.empty_like(x)}
    if op == "gemm":
        dtype, m, n, k = _TORCH[case["dtype"]], case["m"], case["n"], case["k"]
        a = normal(m, k, dtype=dtype)
        b = normal(*((n, k) if case["trans_b"] else (k, n)), dtype=dtype, scale=k ** -0.5)
        return {"case": case, "a": a, "b": b, "c": torch.empty(m, n, device="cuda", dtype=torch.float32 if dtype == torch.bfloat16 else dtype)}
    return {"case": case, "x": (np.random.default_rng(seed).standard_normal((case["outer"], case["reduce"]), dtype=np.float32) * 8)}


def run(state):
    case = state["case"]
    op = case["op"]
    if op in ("mlp", "conv"):
        return state["program"](*state["args"])
    if op == "attention":
        q, k, v, o = state["q"], state["k"], state["v"], state["o"]
        shape = (case["batch"], case["heads"], case["sq"], case["skv"], case["dim"], case["dim"] ** -0.5)
        call = rt.attention_bf16_causal if case["causal"] else rt.attention_bf16
        call(*shape, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), out_bf16=True)
        return o
    if op == "softmax":
        rt.softmax(64 if case["dtype"] == "f64" else 32, case["outer"], case["reduce"], case["inner"], state["x"].data_ptr(), state["y"].data_ptr())
        return state["y"]
    if op == "gemm":
        a, b, c = state["a"], state["b"], state["c"]
        call = {"f64": rt.dgemm, "f32": rt.sgemm, "bf16": rt.bf16gemm_f32}[case["dtype"]]
        call(case["m"], case["n"], case["k"], 1.0, a.data_ptr(), case["k"], b.data_ptr(), b.shape[1], 0.0, c.data_ptr(), case["n"],
             trans_b=rt.TRANS if case["trans_b"] else rt.NO_TRANS)
        return c
    return _softmax_rows(state["x"])


def work(case):
    op = case["op"]
    if op == "mlp":
        t, w = case["tokens"], case["width"]
        return {"bytes": _BYTES[case["dtype"]] * (2 * t * w + 8 * w * w + 8 * w), "flops": 16 * t * w * w}
    if op == "conv":
        n, c, o, size = case["batch"], case["channels"], case["out"], case["size"]
        after = ((size - 1) // case["stride"] + 1) ** 2
        projected = c if case["stride"] != 1 or c != o else 0
        weights = o * (9 * c + 9 * o + projected)
        return {"bytes": 4 * (n * c * size * size + n * o * after + weights), "flops": 2 * n * after * weights}
    if op == "attention":
        pairs, sq, skv, d = case["batch"] * case["heads"], case["sq"], case["skv"], case["dim"]
        seen = sq * (sq + 1) // 2 if case["causal"] else sq * skv
        return {"bytes": 2 * pairs * d * (2 * sq + 2 * skv), "flops": 4 * pairs * d * seen}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        element = _BYTES[case["dtype"]]
        return {"bytes": element * (m * k + k * n) + max(element, 4) * m * n, "flops": 2 * m * n * k}
    n = case["outer"] * case["reduce"] * case.get("inner", 1)
    return {"bytes": 2 * n * _BYTES[case.get("dtype", "f32")], "flops": 0}


def tolerance(case):
    # four times and less what the results were seen to be off from the same operation with everything in 64 bits: bf16 results
    # 2e-3 (the block, with its intermediate values rounded to bf16 too, 2.7e-3), float32 sums 6e-7 over a thousand terms and
    # more over eight thousand, float64 sums 8e-16
    op, dtype = case["op"], case.get("dtype")
    if dtype == "bf16" and op == "mlp":
        return {"rel": 1e-2, "max": 0.05}
    if op == "attention":
        return {"rel": 8e-3, "max": 0.1}
    if dtype == "f64":
        return {"rel": 1e-14, "max": 1e-13}
    return {"rel": 1e-5, "max": 1e-4}
