"""Performance cases of the fused SwiGLU forward: what a program does with this framework, through its torch module.

A case is one call of `fused_mlp_module` on the current stream, on tensors that are already on the GPU:

  op "mlp"         Y = (silu(X @ Wg) * (X @ Wu)) @ Wd   fused_swiglu_mlp_{bf16,fp16}(X, W1W3, W2)
  op "gateup"      H = (X @ Wu) * silu(X @ Wg)          fused_swiglu_{bf16,fp16}(X, W1W3)
  op "gateup_f32"  the same with H in float32           fused_swiglu_bf16_f32out(X, W1W3)
  op "down"        Y = H @ Wd                           swiglu_down_{bf16,fp16}(H, W2)

M is the number of tokens in the call: one token per sequence of the batch when decoding, a prompt (or a chunk of one,
or several packed together) when prefilling. d is the model width, ff the width of the hidden layer.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("fused-swiglu_amd"))

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, op, dtype, M, d, ff):
    return {"name": name, "op": op, "dtype": dtype, "M": M, "d": d, "ff": ff}


def listed():
    return [
        # one token through a small model's layer: the shortest call there is, launches and latency count
        _case("mlp_1_small", "mlp", "bf16", 1, 1024, 2816),
        # one sequence being decoded through an 8B-sized layer: every weight byte is read for one token
        _case("mlp_1", "mlp", "bf16", 1, 4096, 14336),
        # a decode batch of 16 through the same layer
        _case("mlp_16", "mlp", "bf16", 16, 4096, 14336),
        # a larger decode batch, fp16, a 13B-sized layer
        _case("mlp_40_fp16", "mlp", "fp16", 40, 5120, 13824),
        # a short prompt at sizes that are no multiple of any tile
        _case("mlp_200_ragged_fp16", "mlp", "fp16", 200, 3000, 8008),
        # an ordinary prompt through a small layer: few tiles, short K
        _case("mlp_512_small", "mlp", "bf16", 512, 1024, 2816),
        # a short prompt through the 8B-sized layer, an odd number of tokens
        _case("mlp_333", "mlp", "bf16", 333, 4096, 14336),
        # the gate/up operator on its own, a 70B-sized layer, a thousand tokens
        _case("gateup_1000", "gateup", "bf16", 1000, 8192, 28672),
        # its float32 output, a hundred and some tokens (a decode batch of a busy server)
        _case("gateup_f32_130", "gateup_f32", "bf16", 130, 4096, 11008),
        # the down projection on its own, a packed batch of prompts, a 7B-sized layer
        _case("down_2500", "down", "bf16", 2500, 4096, 11008),
        # a long prompt through the 70B-sized layer, fp16
        _case("mlp_2048_fp16", "mlp", "fp16", 2048, 8192, 28672),
        # a full prefill batch through the 8B-sized layer
        _case("mlp_8192", "mlp", "bf16", 8192, 4096, 14336),
    ]


# (d, ff) of the layers the listed cases name; draw() takes one of them or a pair of no such origin
LAYERS = [(1024, 2816), (2048, 8192), (4096, 11008), (4096, 14336), (5120, 13824), (8192, 28672)]
MOST_FLOPS = 6.0 * 8192 * 4096 * 14336  # the largest listed cases


def draw(rng):
    op = rng.choice(["mlp"] * 5 + ["gateup"] * 3 + ["gateup_f32", "down"])
    dtype = "bf16" if op == "gateup_f32" else rng.choice(["bf16", "bf16", "fp16"])
    if rng.random() < 0.5:
        d, ff = rng.choice(LAYERS)
    else:  # any width: the entry points take multiples of 8
        d = 8 * round(math.exp(rng.uniform(math.log(1024), math.log(8192))) / 8)
        ff = 8 * round(d * rng.uniform(2.5, 4.0) / 8)
    M = round(math.exp(rng.uniform(0.0, math.log(8192))))
    M = max(1, min(M, int(MOST_FLOPS / (6.0 * d * ff))))
    return {"op": op, "dtype": dtype, "M": M, "d": d, "ff": ff}


def _tensors(case, seed):
    """Activations ~ N(0, 1) (half of that in fp16, whose range is short), weights ~ N(0, 1) / sqrt(fan_in): values of a
    trained layer's size. H of the down projection alone has the spread that a gated product of such values has."""
    M, d, ff, dtype = case["M"], case["d"], case["ff"], DTYPES[case["dtype"]]
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    x_scale = 0.5 if case["dtype"] == "fp16" else 1.0

    def normal(rows, cols, scale):
        t = torch.empty((rows, cols), dtype=dtype, device=dev)
        return t.normal_(0.0, scale, generator=g)

    if case["op"] == "down":
        up, gate = normal(M, ff, x_scale), normal(M, ff, x_scale)
        return up * torch.nn.functional.silu(gate), normal(d, ff, ff ** -0.5)
    args = (normal(M, d, x_scale), normal(2 * ff, d, d ** -0.5))
    return args + (normal(d, ff, ff ** -0.5),) if case["op"] == "mlp" else args


def prepare(case, seed):
    """The activations and the weights, as a layer of the program holds them, and the entry point it calls."""
    import fused_mlp_module
    name = {"mlp": "fused_swiglu_mlp_" + case["dtype"], "gateup": "fused_swiglu_" + case["dtype"],
            "gateup_f32": "fused_swiglu_bf16_f32out", "down": "swiglu_down_" + case["dtype"]}[case["op"]]
    return {"fn": getattr(fused_mlp_module, name), "args": _tensors(case, seed)}


def run(state):
    return state["fn"](*state["args"])


def work(case):
    """Inputs once, output once (H stays inside "mlp"), and the products' multiplications and additions."""
    M, d, ff = case["M"], case["d"], case["ff"]
    if case["op"] == "mlp":
        return {"bytes": 2 * (3 * d * ff + 2 * M * d), "flops": 6 * M * d * ff}
    if case["op"] == "down":
        return {"bytes": 2 * (d * ff + M * ff + M * d), "flops": 2 * M * d * ff}
    out = 4 if case["op"] == "gateup_f32" else 2
    return {"bytes": 2 * (2 * d * ff + M * d) + out * M * ff, "flops": 4 * M * d * ff}


def tolerance(case):
    """Against the same formula in float64, on the listed sizes: one rounding of the result to bf16 is rel 1.7e-3, max
    3.9e-3; with H rounded in between 2.4e-3 and up to 1.0e-2; fp16 is an eighth of that (2.9e-4 and 1.2e-3 with H
    rounded); fp32 sums of 4096 products in float32 are 6e-7 and 7e-6. Four times these."""
    if case["op"] == "gateup_f32":
        return {"rel": 5e-6, "max": 5e-5}
    if case["op"] == "mlp":
        return {"rel": 1e-2, "max": 4e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 5e-3}
    return {"rel": 7e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 8e-4, "max": 2e-3}


def exact(case, seed):
    """The formulas in float64: rows 2j of W1W3 are the up operand, rows 2j + 1 the gate."""
    args = [t.double() for t in _tensors(case, seed)]
    if case["op"] == "down":
        return args[0] @ args[1].t()
    pre = args[0] @ args[1].t()
    up, gate = pre[:, 0::2], pre[:, 1::2]
    h = up * (gate / (1.0 + torch.exp(-gate)))
    return h @ args[2].t() if case["op"] == "mlp" else h
