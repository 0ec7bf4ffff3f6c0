"""The work that programs have this package do, as cases that can be timed: linear layers on FP8 weights from one decoded
token to a full prefill, mixture-of-experts feed-forward layers through the three grouped entry points, the grouped weight
gradient of their training, and rows that are stored as FP8 and read back.

A case is a dict of plain values; `prepare` makes what a program holds before the call, `run` is one pass through the
public entry points.  Activations are bf16 N(0, 1) with one channel in a hundred scaled by 20 (the outliers that row scales
exist for), weights N(0, 0.02), both as in mslk_amd/workloads.py.
"""
from __future__ import annotations

import math

import torch

import mslk_amd

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _linear(m, n, k, layout="rows", bias="", out="bf16", one_call=False):
    return {"kind": "linear", "m": m, "n": n, "k": k, "layout": layout, "bias": bias, "out": out, "one_call": one_call}


def _moe(experts, rows, d, f, api):
    return {"kind": "moe", "experts": experts, "rows": rows, "d": d, "f": f, "api": api}


def _weight_grad(experts, rows, m, n):
    return {"kind": "weight_grad", "experts": experts, "rows": rows, "m": m, "n": n}


def _rows(rows, k, dtype):
    return {"kind": "rows", "rows": rows, "k": k, "dtype": dtype}


def listed():
    named = {
        # One decoded token through a square projection: activations are quantized and multiplied in one call.
        "decode_1": _linear(1, 8192, 8192, one_call=True),
        # A small decode batch through the same projection, quantizer and product as two calls.
        "decode_16": _linear(16, 8192, 8192),
        # A larger decode batch through a down projection whose weights were pre-shuffled when the model was loaded.
        "decode_64_preshuffled": _linear(64, 4096, 14336, layout="preshuffled"),
        # A small layer (or a small model) at a moderate batch: launches count.
        "linear_1024": _linear(1024, 1024, 1024),
        # A chunk of a prompt through a fused query/key/value projection: a few hundred rows, no round number.
        "prefill_500": _linear(500, 10240, 8192),
        # The square product that the benchmark is quoted on, with the quantizer in front of it.
        "linear_4096": _linear(4096, 4096, 4096),
        # A full prefill through a fused gate and up projection with a bias.
        "prefill_8192_bias": _linear(8192, 28672, 4096, bias="bf16"),
        # Sixteen large experts in prefill; the program knows the group sizes and passes lists of tensors.
        "moe_16_prefill": _moe(16, 8192, 5120, 4096, "list"),
        # The same layer decoding: a few rows per expert, sizes on the GPU only.
        "moe_16_decode": _moe(16, 256, 5120, 4096, "stacked"),
        # Many small experts, thousands of routed rows, cumulative offsets on the GPU.
        "moe_128_prefill": _moe(128, 32768, 2048, 768, "offsets"),
        # The weight gradient of an expert layer in training: the contraction runs over each expert's rows, which the
        # program pads to a multiple of 16 as FP8 training does.
        "moe_weight_grad": _weight_grad(8, 16384, 4096, 2048),
        # A key/value cache stored as FP8, one scale per head and token, and read back: rows of one head.
        "cache_rows_128": _rows(131072, 128, "bf16"),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


_DIMS = (1024, 1536, 2048, 2560, 3072, 3584, 4096, 5120, 6144, 7168, 8192, 10240, 11008, 13824, 14336, 16384, 22016, 28672)


def _popularity(experts):
    weight = [(rank + 1.0) ** -1.1 for rank in range(experts)]
    return [w / sum(weight) for w in weight]


def _used_experts(experts, rows):
    """How many experts get a row at all, on average: the others' weights need not be read."""
    return sum(1.0 - (1.0 - p) ** rows for p in _popularity(experts))


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 2.5e15)


def draw(rng):
    most = {}
    for case in listed():
        most[case["kind"]] = max(most.get(case["kind"], 0.0), _cost(case))
    kind = rng.choice(("linear", "linear", "linear", "moe", "moe", "weight_grad", "rows"))
    while True:
        if kind == "linear":
            m, n, k = _log(rng, 1, 8192), rng.choice(_DIMS), rng.choice(_DIMS)
            layout = rng.choice(("rows", "rows", "rows", "preshuffled"))
            if layout == "rows" and rng.random() < 0.2:   # a head whose width is no round number
                n += rng.randrange(1, 512)
            one_call = layout == "rows" and m <= 4
            case = _linear(m, n, k, layout, rng.choice(("", "", "bf16", "fp32")),
                           "bf16" if one_call else rng.choice(("bf16", "bf16", "bf16", "fp16")), one_call)
        elif kind == "moe":
            case = _moe(rng.choice((8, 16, 32, 64, 128)), _log(rng, 64, 32768), rng.choice((1024, 2048, 2880, 4096, 5120, 7168)),
                        rng.choice((768, 1024, 1408, 2048, 2880, 4096)), rng.choice(("list", "stacked", "offsets")))
        elif kind == "weight_grad":
            case = _weight_grad(rng.choice((4, 8, 16, 32)), _log(rng, 2048, 32768) // 16 * 16,
                                rng.choice((1024, 1408, 2048, 2880, 4096, 5120)), rng.choice((1024, 1408, 2048, 2880, 4096)))
        else:
            case = _rows(_log(rng, 64, 262144), rng.choice((64, 80, 96, 128, 192, 256, 512, 576, 1024, 4096)),
                         rng.choice(("bf16", "bf16", "fp16", "fp32")))
        if _cost(case) <= most[kind]:
            return case


def _activations(gen, rows, cols, dtype=torch.bfloat16):
    x = torch.randn(rows, cols, generator=gen, device="cuda", dtype=dtype)
    loud = torch.randperm(cols, generator=gen, device="cuda")[: cols // 100]
    x[:, loud] *= 20
    return x


def _weights(gen, *shape):
    """Codes and row scales of N(0, 0.02) weights, quantized once as when a model is loaded."""
    w = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.02)
    return mslk_amd.quantize_fp8_row(w)


def _group_sizes(gen, experts, rows, multiple=1):
    """Rows per expert under a popularity that falls like 1 / rank^1.1, the popular experts anywhere."""
    share = torch.tensor(_popularity(experts), dtype=torch.float64, device="cuda")
    share = share[torch.randperm(experts, generator=gen, device="cuda")]
    hits = torch.multinomial(share, rows // multiple, replacement=True, generator=gen)
    return torch.bincount(hits, minlength=experts) * multiple


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        n, k = case["n"], case["k"]
        s["x"] = _activations(gen, case["m"], k)
        s["wq"], s["ws"] = _weights(gen, n, k)
        if case["layout"] == "preshuffled":
            s["wq"] = mslk_amd.preshuffle_b_mfma(s["wq"])
        s["bias"] = None
        if case["bias"]:
            s["bias"] = (torch.randn(n, generator=gen, device="cuda") * 0.01).to(_DTYPES[case["bias"]])
    elif kind == "moe":
        experts, rows, d, f = case["experts"], case["rows"], case["d"], case["f"]
        sizes = _group_sizes(gen, experts, rows)
        s["x"] = _activations(gen, rows, d)
        # rows in expert order and where each comes from: a router's answer
        s["tokens"] = torch.randperm(rows, generator=gen, device="cuda").to(torch.int32)
        s["owner"] = torch.repeat_interleave(torch.arange(experts, device="cuda"), sizes).to(torch.int32)
        s["scores"] = torch.rand(rows, experts, generator=gen, device="cuda")
        s["w13"], s["s13"] = _weights(gen, experts, 2 * f, d)
        s["w2"], s["s2"] = _weights(gen, experts, d, f)
        if case["api"] == "list":
            s["sizes"] = sizes.tolist()
            for name in ("w13", "s13", "w2", "s2"):
                s[name] = list(s[name].unbind(0))
        elif case["api"] == "stacked":
            s["sizes"] = sizes
        else:
            s["offsets"] = sizes.cumsum(0).to(torch.int32)
    elif kind == "weight_grad":
        experts, rows = case["experts"], case["rows"]
        sizes = _group_sizes(gen, experts, rows, 16)
        s["offsets"] = sizes.cumsum(0).to(torch.int32)
        for name, side in (("g", case["m"]), ("x", case["n"])):
            codes, scales, begin = [], [], 0
            t = _activations(gen, rows, side).t()
            for size in sizes.tolist():
                q, q_scale = mslk_amd.quantize_fp8_row(t[:, begin:begin + size]) if size else (
                    t.new_empty(side, 0, dtype=mslk_amd.FP8_DTYPE), torch.ones(side, device="cuda"))
                codes.append(q)
                scales.append(q_scale)
                begin += size
            s[name], s[name + "_scale"] = torch.cat(codes, 1), torch.cat(scales)
        s["grad"] = torch.empty(experts, case["m"], case["n"], dtype=torch.bfloat16, device="cuda")
    else:
        s["x"] = _activations(gen, case["rows"], case["k"], _DTYPES[case["dtype"]])
    return s


def _run_linear(s):
    case = s["case"]
    if case["one_call"]:
        return torch.ops.mslk.quantize_f8f8bf16_rowwise(s["x"], s["wq"], s["ws"], s["bias"])
    xq, xs = mslk_amd.quantize_fp8_row(s["x"])
    if case["layout"] == "preshuffled":
        op = torch.ops.mslk.f8f8f16_rowwise_preshuffle if case["out"] == "fp16" else torch.ops.mslk.f8f8bf16_rowwise_preshuffle
    else:
        op = torch.ops.mslk.f8f8f16_rowwise if case["out"] == "fp16" else torch.ops.mslk.f8f8bf16_rowwise
    return op(xq, s["wq"], xs, s["ws"], s["bias"])


def _grouped(s, xq, xs, w, w_scale):
    api = s["case"]["api"]
    if api == "list":
        return torch.ops.mslk.f8f8bf16_rowwise_grouped_cat(list(xq.split(s["sizes"])), w, list(xs.split(s["sizes"])), w_scale)
    if api == "stacked":
        return torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, w, xs, w_scale, s["sizes"])
    y = torch.empty(xq.shape[0], w.shape[1], dtype=torch.bfloat16, device=xq.device)
    return torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xq, w, xs, w_scale, s["offsets"], y)


def _run_moe(s):
    f = s["case"]["f"]
    xq, xs = mslk_amd.gather_scale_quant_dense_tokens(s["x"], s["tokens"], s["owner"], s["scores"])
    h = _grouped(s, xq, xs, s["w13"], s["s13"])
    aq, a_scale = mslk_amd.silu_mul_quant(h[:, :f], h[:, f:])
    return _grouped(s, aq, a_scale, s["w2"], s["s2"])


def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        return _run_linear(state)
    if kind == "moe":
        return _run_moe(state)
    if kind == "weight_grad":
        return torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(state["g"], state["x"], state["g_scale"], state["x_scale"],
                                                          state["offsets"], state["grad"])
    xq, xs = mslk_amd.quantize_fp8_row(state["x"])
    return xq, xs, mslk_amd.dequantize_fp8_row(xq, xs)


def work(case):
    """Inputs once, outputs once; what passes between the calls of a pass is not counted."""
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        codes = m * k + 4 * m if case["one_call"] else 0   # this call returns the codes and scales as well
        return {"bytes": 2 * m * k + n * k + 2 * m * n + 4 * n + codes, "flops": 2 * m * n * k}
    if kind == "moe":
        experts, rows, d, f = case["experts"], case["rows"], case["d"], case["f"]
        used = _used_experts(experts, rows)
        return {"bytes": 2 * rows * d + 12 * rows + used * (3 * f * d + 4 * (2 * f + d)) + 2 * rows * d, "flops": 6 * rows * d * f}
    if kind == "weight_grad":
        experts, rows, m, n = case["experts"], case["rows"], case["m"], case["n"]
        return {"bytes": rows * (m + n) + 4 * experts * (m + n) + 2 * experts * m * n, "flops": 2 * rows * m * n}
    rows, k = case["rows"], case["k"]
    size = {"bf16": 2, "fp16": 2, "fp32": 4}[case["dtype"]]
    return {"bytes": rows * (k * (size + 3) + 4), "flops": 0}


def tolerance(case):
    """Codes, scales and their bf16 products are fixed bit for bit.  A matrix product is summed in fp32 and rounded once: set
    beside the same codes multiplied in 64 bits it shows 1.7e-3 in bf16 and 2.1e-4 in fp16, at most 4.1e-3 and 5.7e-4 of one
    value, and 7.8e-3 (one bf16 step) beside the same sums in another order.  The expert layer quantizes an intermediate
    result again, where a value next to a rounding boundary may land on the other side of it: with that activation in 64 bits
    3.3e-3 over all, up to 0.25 of one value (a flipped code of a channel that dominates its row)."""
    if case["kind"] == "rows":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 1.3e-2, "max": 0.8}
    if case.get("out") == "fp16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 6.5e-3, "max": 1.6e-2}
