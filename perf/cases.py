"""The calls this runtime is timed at: the seven templates through the Python
binding, each from its smallest everyday call to its largest, with the ragged
sizes that real programs bring.

Inputs are torch tensors on the GPU and the calls go to the null stream, which
is torch's own, as a program that mixes the two would make them. Everything
is fp32: the templates take no other type.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "kernel.h_amd"))
import kernelh as kh  # noqa: E402

HEAD_DIM = 64  # attention is pinned to it


def listed():
    return [
        # The smallest call: one launch of a few workgroups, where what the
        # call costs is its latency. Odd, as the smoke test has it.
        {"name": "vecadd_4099", "op": "vecadd", "n": 4099},
        # An activation over a mid-sized layer's output (benchmark size).
        {"name": "gelu_2e22", "op": "fused_gelu", "n": 1 << 22},
        # Attention-score rows (benchmark size).
        {"name": "softmax_4096x1024", "op": "softmax", "rows": 4096, "cols": 1024},
        # Rows over a large set of classes: few rows, each tens of thousands
        # of floats, and a count that is no multiple of anything.
        {"name": "softmax_256x32001", "op": "softmax", "rows": 256, "cols": 32001},
        # Normalisation of a wide layer: rows past one wave's registers.
        {"name": "layernorm_2048x5000", "op": "layernorm", "rows": 2048, "cols": 5000},
        # Prefix sums: one round of workgroups, and the largest (both
        # benchmark sizes).
        {"name": "scan_1e6", "op": "scan", "n": 1000000},
        {"name": "scan_2e26", "op": "scan", "n": 1 << 26},
        # A weight matrix applied to a handful of rows (small-batch
        # inference): bound by reading the weights.
        {"name": "gemm_16x4096x4096", "op": "gemm", "m": 16, "n": 4096, "k": 4096},
        # A product whose extents come from data: all three odd or ragged.
        {"name": "gemm_1000x1003x999", "op": "gemm", "m": 1000, "n": 1003, "k": 999},
        # The largest product (the headline benchmark size).
        {"name": "gemm_8192", "op": "gemm", "m": 8192, "n": 8192, "k": 8192},
        # Attention over a whole batch (benchmark size), and of one short
        # sequence of no particular length, which leaves most of the chip to fill.
        {"name": "attention_b4h16s1024", "op": "attention", "batch": 4, "heads": 16, "seq": 1024},
        {"name": "attention_b1h8s777", "op": "attention", "batch": 1, "heads": 8, "seq": 777},
    ]


def _spread(rng, lo, hi, step=1):
    """A size from lo to hi, spread over its logarithm; a multiple of `step`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v // step * step))


def draw(rng):
    op = rng.choice(["vecadd", "fused_gelu", "softmax", "layernorm", "scan", "gemm", "gemm", "attention"])
    # Half of the sizes are whole multiples of 16 and half are whatever comes.
    step = rng.choice([1, 16])
    if op in ("vecadd", "fused_gelu", "scan"):
        return {"op": op, "n": _spread(rng, 1024, 1 << 26, step)}
    if op in ("softmax", "layernorm"):
        cols = _spread(rng, 64, 65536, step)
        return {"op": op, "rows": _spread(rng, 16, min(32768, (1 << 26) // cols)), "cols": cols}
    if op == "gemm":
        # m is the batch side (from one row), n and k the layer's; at most
        # half the work of the largest listed product.
        m, n, k = _spread(rng, 1, 8192), _spread(rng, 64, 8192, step), _spread(rng, 64, 8192, step)
        while m * n * k > 1 << 37:
            m //= 2
        return {"op": op, "m": m, "n": n, "k": k}
    return {"op": op, "batch": rng.randint(1, 4), "heads": rng.choice([1, 2, 4, 6, 8, 12, 16]),
            "seq": _spread(rng, 64, 4096, step)}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(g, n, lo=-1.0, hi=1.0):
    return torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo


def _normal(g, n, sd=1.0):
    return torch.randn(n, generator=g, device="cuda") * sd


def _inputs(case, seed):
    g = _generator(seed)
    op = case["op"]
    if op == "vecadd":
        return [_uniform(g, case["n"]), _uniform(g, case["n"])]
    if op == "fused_gelu":
        return [_normal(g, case["n"])]
    if op == "softmax":
        return [_normal(g, case["rows"] * case["cols"], 4.0)]
    if op == "layernorm":
        c = case["cols"]
        return [_normal(g, case["rows"] * c, 4.0), _uniform(g, c, 0.5, 1.5), _uniform(g, c, -0.1, 0.1)]
    if op == "scan":
        return [torch.rand(case["n"], generator=g, device="cuda")]  # the 2^-24 grid: every prefix is exact in 64 bits
    if op == "gemm":
        return [_uniform(g, case["m"] * case["k"]), _uniform(g, case["k"] * case["n"])]
    n = case["batch"] * case["heads"] * case["seq"] * HEAD_DIM
    return [_normal(g, n), _normal(g, n), _normal(g, n)]


def _out_shape(case):
    op = case["op"]
    if op in ("softmax", "layernorm"):
        return case["rows"], case["cols"]
    if op == "gemm":
        return case["m"], case["n"]
    if op == "attention":
        return case["batch"], case["heads"], case["seq"], HEAD_DIM
    return (case["n"],)


def prepare(case, seed):
    """The inputs, the output buffer and, for the scan, its workspace."""
    x = _inputs(case, seed)
    out = torch.empty(_out_shape(case), device="cuda")
    p = [t.data_ptr() for t in x]
    y = out.data_ptr()
    keep = []
    op = case["op"]
    if op == "vecadd":
        args = (p[0], p[1], y, case["n"])
    elif op == "fused_gelu":
        args = (p[0], None, y, case["n"])
    elif op == "softmax":
        args = (p[0], y, case["rows"], case["cols"])
    elif op == "layernorm":
        args = (p[0], p[1], p[2], y, case["rows"], case["cols"])
    elif op == "scan":
        keep = [torch.zeros(kh.scan_workspace_floats(case["n"]), device="cuda") for _ in range(2)]
        args = (p[0], y, None, keep[0].data_ptr(), keep[1].data_ptr(), case["n"])
    elif op == "gemm":
        args = (p[0], p[1], y, case["m"], case["n"], case["k"])
    else:
        args = (p[0], p[1], p[2], y, case["batch"], case["heads"], case["seq"], HEAD_DIM)
    return {"call": getattr(kh, op), "args": args, "out": out, "keep": (x, keep)}


def run(state):
    state["call"](*state["args"])
    return state["out"]


def work(case):
    op = case["op"]
    if op == "vecadd":
        return {"bytes": 12 * case["n"], "flops": case["n"]}
    if op == "fused_gelu":
        return {"bytes": 8 * case["n"], "flops": 12 * case["n"]}
    if op == "softmax":
        e = case["rows"] * case["cols"]
        return {"bytes": 8 * e, "flops": 5 * e}
    if op == "layernorm":
        e = case["rows"] * case["cols"]
        return {"bytes": 8 * e + 8 * case["cols"], "flops": 8 * e}
    if op == "scan":
        return {"bytes": 8 * case["n"], "flops": case["n"]}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    e = case["batch"] * case["heads"] * case["seq"]
    return {"bytes": 16 * e * HEAD_DIM, "flops": 4 * e * case["seq"] * HEAD_DIM}


def tolerance(case):
    # vecadd is one IEEE addition and the scan's prefixes are exact in 64 bits
    # before their one rounding: both have one right answer. The others are
    # about four times the largest error measured against 64 bits: products
    # 1.6e-6 (sums of up to 8192 terms in 32 bits, in any order), rows of
    # exponentials 1e-6 (the rounding of an exponent of a few tens), the rest
    # below 3e-7.
    if case["op"] in ("vecadd", "scan"):
        return "exact"
    rel = {"gemm": 6e-6, "softmax": 4e-6, "attention": 4e-6}.get(case["op"], 1e-6)
    return {"rel": rel, "max": 40 * rel}


def exact(case, seed):
    x = [t.double() for t in _inputs(case, seed)]
    op = case["op"]
    if op == "vecadd":
        return x[0] + x[1]
    if op == "fused_gelu":
        t = 1.5 * x[0] + 0.5
        return 0.5 * t * (1 + torch.tanh(0.7978845608 * (t + 0.044715 * t ** 3)))
    if op == "softmax":
        return torch.softmax(x[0].view(_out_shape(case)), dim=1)
    if op == "layernorm":
        r = x[0].view(_out_shape(case))
        d = r - r.mean(dim=1, keepdim=True)
        return d * torch.rsqrt((d * d).mean(dim=1, keepdim=True) + 1e-5) * x[1] + x[2]
    if op == "scan":
        return torch.cumsum(x[0], dim=0)
    if op == "gemm":
        return x[0].view(case["m"], case["k"]) @ x[1].view(case["k"], case["n"])
    b, h, s, d = _out_shape(case)
    q, k, v = (t.view(b * h, s, d) for t in x)
    out = torch.empty(b * h, s, d, dtype=torch.float64, device="cuda")
    for i in range(b * h):
        out[i] = torch.softmax((q[i] @ k[i].T.contiguous()) / math.sqrt(d), dim=1) @ v[i]
    return out.view(b, h, s, d)
