"""The work that programs have this library do, as timed cases: dense products, the gated feed-forward block, conv2d.

A case is a dict of plain values.  ``listed()`` names twelve of them, ``draw(rng)`` gives one more of the same ranges,
``prepare`` makes on the GPU what a program holds before the call (activations, weights), ``run`` makes the one call
through the public entry points and returns its whole result, ``work`` states the bytes and operations the call cannot
do without, ``tolerance`` how far another correct implementation at the same precision may be off.

The ranges: products with m from 1 to 8192 rows, n and k from 64 to 28672, in bfloat16, float16, int8 (int32 result) and
float32, row-major ("nn"), with a transposed weight ("nt": ``x @ w.t()``) and with a transposed left operand ("tn":
``x.t() @ dy``); feed-forward blocks of 1 to 4096 rows over widths 512 to 4096 and up to 14336 hidden units; conv2d
forward of filters 1x1 to 5x5, strides 1 and 2, planes of 7 to 112 pixels a side, 3 to 2048 channels, 1 to 128 images.
No case is larger than the largest listed one.
"""
import math
import os

import torch

# The library's own choice of tile, no search per size: a program that meets new sizes all the time (sequence lengths,
# batch sizes) runs this way, since a search takes tens of seconds for every new size.
os.environ["TRITONIX_AUTOTUNE"] = "0"

import tritonix  # noqa: E402
from tritonix.ops.conv2d import conv2d_forward  # noqa: E402
from tritonix.ops.matmul import matmul_splitk  # noqa: E402
from tritonix.ops.swiglu import glu, swiglu_ffn  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8, "f32": torch.float32}
SIZES = {"bf16": 2, "f16": 2, "i8": 1, "f32": 4}

MOST_FLOPS = 2.0 * 8192 ** 3
MOST_BYTES = 4.0e8


def listed():
    return [
        # the smallest call: a small float16 product, bound by launch latency
        dict(name="matmul_f16_small", op="matmul", dtype="f16", layout="nn", m=1024, n=768, k=512),
        # one decode step of a 16-sequence batch through a down-projection: the weight is streamed once
        dict(name="splitk_bf16_decode", op="splitk", dtype="bf16", layout="nn", m=16, n=4096, k=14336),
        # a linear layer with an [out, in] weight on a medium batch of rows
        dict(name="matmul_bf16_linear", op="matmul", dtype="bf16", layout="nt", m=512, n=4096, k=4096),
        # sizes that no tile divides, rows that are not 16-byte aligned
        dict(name="matmul_bf16_ragged", op="matmul", dtype="bf16", layout="nn", m=1025, n=2050, k=4100),
        # the weight gradient of a linear layer: x.t() @ dy
        dict(name="matmul_bf16_wgrad", op="matmul", dtype="bf16", layout="tn", m=4096, n=4096, k=2048),
        # float32 operands, as the numerical parts of a program have them
        dict(name="matmul_f32", op="matmul", dtype="f32", layout="nn", m=2048, n=2048, k=2048),
        # the large square products of both matrix types: the largest calls
        dict(name="matmul_bf16_large", op="matmul", dtype="bf16", layout="nn", m=8192, n=8192, k=8192),
        dict(name="matmul_i8_large", op="matmul", dtype="i8", layout="nn", m=8192, n=8192, k=8192),
        # the feed-forward block: prefill of 4096 tokens, and a decode step of 16
        dict(name="ffn_bf16_prefill", op="ffn", dtype="bf16", act="silu", m=4096, d=4096, h=14336),
        dict(name="ffn_bf16_decode", op="ffn", dtype="bf16", act="silu", m=16, d=4096, h=14336),
        # convolution layers of an image network: 3x3 on large planes, and the 3x3 stride-2 layer between two stages
        dict(name="conv_bf16_3x3", op="conv", dtype="bf16", batch=32, c_in=256, c_out=256, hw=56, f=3, stride=1, pad=1, dil=1),
        dict(name="conv_f16_stride2", op="conv", dtype="f16", batch=32, c_in=128, c_out=128, hw=56, f=3, stride=2, pad=1, dil=1),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]: of every ten, six multiples of 64, two of 8, two as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    unit = rng.choice([64] * 6 + [8] * 2 + [1] * 2)
    return min(max(lo, (v + unit // 2) // unit * unit), hi) if v >= unit else v


def _drawn(rng):
    op = rng.choice(["matmul"] * 5 + ["splitk", "glu", "ffn", "conv", "conv", "conv"])
    if op == "matmul":
        return dict(op=op, dtype=rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "i8", "i8", "f32"]),
                    layout=rng.choice(["nn", "nn", "nn", "nt", "nt", "tn"]),
                    m=_log_int(rng, 1, 8192), n=_log_int(rng, 64, 28672), k=_log_int(rng, 64, 14336))
    if op == "splitk":
        return dict(op=op, dtype=rng.choice(["bf16", "f16", "i8"]), layout=rng.choice(["nn", "nt"]), m=_log_int(rng, 1, 64),
                    n=_log_int(rng, 512, 28672), k=_log_int(rng, 1024, 14336))
    if op == "glu":
        return dict(op=op, dtype=rng.choice(["bf16", "f16"]), act=rng.choice(["silu", "sigmoid"]), m=_log_int(rng, 1, 4096),
                    d=_log_int(rng, 512, 4096), h=_log_int(rng, 512, 14336))
    if op == "ffn":
        return dict(op=op, dtype=rng.choice(["bf16", "f16"]), act="silu", m=_log_int(rng, 1, 4096), d=_log_int(rng, 512, 4096),
                    h=_log_int(rng, 512, 14336))
    f = rng.choice([1, 1, 3, 3, 3, 5])
    most = 2048 if f == 1 else 512
    return dict(op=op, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), batch=rng.choice([1, 4, 8, 16, 32, 64, 128]),
                c_in=3 if rng.random() < 0.1 else _log_int(rng, 16, most), c_out=_log_int(rng, 16, most),
                hw=rng.choice([7, 14, 17, 28, 33, 56, 112]), f=f, stride=rng.choice([1, 1, 1, 2]), pad=f // 2,
                dil=1)


def draw(rng):
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


def _out_hw(c):
    return (c["hw"] + 2 * c["pad"] - c["dil"] * (c["f"] - 1) - 1) // c["stride"] + 1


def work(case):
    """Operands read once, the result written once; two operations per multiply-add."""
    c, s = case, SIZES[case["dtype"]]
    if c["op"] in ("matmul", "splitk"):
        out = 4 if c["dtype"] == "i8" else s
        return {"bytes": float(s * (c["m"] * c["k"] + c["k"] * c["n"]) + out * c["m"] * c["n"]),
                "flops": 2.0 * c["m"] * c["n"] * c["k"]}
    if c["op"] == "glu":
        return {"bytes": float(s * (c["m"] * c["d"] + 2 * c["d"] * c["h"] + c["m"] * c["h"])), "flops": 4.0 * c["m"] * c["d"] * c["h"]}
    if c["op"] == "ffn":
        return {"bytes": float(s * (2 * c["m"] * c["d"] + 3 * c["d"] * c["h"])), "flops": 6.0 * c["m"] * c["d"] * c["h"]}
    o = _out_hw(c)
    taps = c["c_in"] * c["f"] * c["f"]
    return {"bytes": float(s * (c["batch"] * c["c_in"] * c["hw"] ** 2 + c["c_out"] * (taps + 1) + c["batch"] * c["c_out"] * o * o)),
            "flops": 2.0 * c["batch"] * o * o * c["c_out"] * taps}


def _normal(shape, dtype, scale, gen):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, scale, generator=gen).to(dtype)


def _matrix(rows, cols, dtype, scale, gen, transposed):
    """A [rows, cols] operand, row-major or as the transposed view of a row-major [cols, rows] one."""
    shape = (cols, rows) if transposed else (rows, cols)
    if dtype == torch.int8:
        t = torch.empty(shape, dtype=dtype, device="cuda").random_(-127, 128, generator=gen)
    else:
        t = _normal(shape, dtype, scale, gen)
    return t.t() if transposed else t


def prepare(case, seed):
    c, dtype = case, DTYPES[case["dtype"]]
    gen = torch.Generator("cuda").manual_seed(int(seed))
    state = {"case": dict(case)}
    if c["op"] in ("matmul", "splitk"):
        state["a"] = _matrix(c["m"], c["k"], dtype, 1.0, gen, c["layout"] == "tn")
        state["b"] = _matrix(c["k"], c["n"], dtype, 1.0 / math.sqrt(c["k"]), gen, c["layout"] == "nt")
    elif c["op"] in ("glu", "ffn"):
        # gate and linear weights interleaved column-wise, as the fused kernel takes them
        state["x"] = _normal((c["m"], c["d"]), dtype, 1.0, gen)
        state["w12"] = _normal((c["d"], 2 * c["h"]), dtype, 0.02, gen)
        if c["op"] == "ffn":
            state["w3"] = _normal((c["h"], c["d"]), dtype, 0.02, gen)
    else:
        fan_in = c["c_in"] * c["f"] * c["f"]
        state["x"] = _normal((c["batch"], c["c_in"], c["hw"], c["hw"]), dtype, 1.0, gen)
        state["w"] = _normal((c["c_out"], c["c_in"], c["f"], c["f"]), dtype, 1.0 / math.sqrt(fan_in), gen)
        state["bias"] = _normal((c["c_out"],), dtype, 1.0, gen)
    return state


def run(state):
    c = state["case"]
    if c["op"] == "matmul":
        return tritonix.matmul(state["a"], state["b"])
    if c["op"] == "splitk":
        return matmul_splitk(state["a"], state["b"])
    if c["op"] == "glu":
        return glu(state["x"], state["w12"], activation=c["act"])
    if c["op"] == "ffn":
        return swiglu_ffn(state["x"], state["w12"], state["w3"], activation=c["act"])
    return conv2d_forward(state["x"], state["w"], state["bias"], (c["stride"], c["stride"]), (c["pad"], c["pad"]),
                          (c["dil"], c["dil"]))


def tolerance(case):
    """Four times what the results were measured to be off the same product in 64 bits (the rounding of the result; for
    the gated products that of the intermediate too; for float32 the matrix instructions' three-term split)."""
    if case["dtype"] == "i8":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 1.8e-5, "max": 1e-4}
    rel = {"bf16": 7e-3, "f16": 9e-4}[case["dtype"]]
    if case["op"] in ("glu", "ffn"):
        return {"rel": 1.5 * rel, "max": 6 * rel}
    return {"rel": rel, "max": 2.5 * rel}
