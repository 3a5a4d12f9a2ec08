"""The work that the performance of this package is measured on: whole calls of its public entry points, at the sizes
the FLUX and SDXL drivers run them with.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program has in hand before the call: activations, the converted layer, the row list
    run(state)           one pass, as a program makes it
    work(case)           bytes and operations a pass cannot do without
    tolerance(case)      how far another correct implementation may be
    exact(case, seed)    the same outputs in 64 bits, from plain torch

Kinds of case:
    layer    y = Int8Linear(x): per-token quantizer (+ low-rank down-projection), fused INT8 GEMM, dequant, bias
    split    y = SplitInLinear(x): FLUX's single-block proj_out cut at 3072, both halves Int8Linear with a low-rank
             branch of their own, the second summed into the first
    routed   the routed executor's layer: the active tokens' rows gathered into the quantizer, the results scattered
             into the cached canvas
    convert  Int8Linear(lin): the weight's round-to-nearest codes, scales and kernel layout, once per layer at load

Activations are N(0, 1) with 0.5 % of the channels 20 times larger (the outlier channels of the benchmark's
workloads), weights N(0, 0.02), low-rank factors N(0, 0.02), bias N(0, 0.01).
"""
import math

import torch
import torch.nn as nn

from pyraquant_amd.int8_exec import (FLUX_TOKEN_SHAPES, LOWRANK_A_ATTR, LOWRANK_B_ATTR, Int8Linear,
                                     convert_linears_to_int8)
from pyraquant_amd.routing import leaf_mask, routed_row_index
from pyraquant_amd.sdxl import SDXL_TOKEN_SHAPES, SdxlInt8Linear
from pyraquant_amd.weights import SplitInLinear

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
GRID = 256                       # packed tokens along an edge of a 4096 x 4096 image
SPLIT_AT = 3072                  # FLUX's single-block proj_out: attention (3072) and MLP (12288) inputs
MOST = 65536 * 3072 * 12288      # multiply-adds of the largest listed case


def _layer(name, M, K, N, dtype="bf16", rank=0, group=0, bias=True):
    return {"name": name, "kind": "layer", "M": M, "K": K, "N": N, "dtype": dtype, "rank": rank, "group": group,
            "bias": bias}


def listed():
    return [
        # SDXL cross-attention key / value projection: two prompts of 77 text tokens; the smallest call there is
        _layer("sdxl_text_kv", 154, 2048, 1280, "fp16", bias=False),
        # SDXL 1K stage, attention output projection of the 1280-channel blocks (2 x 1024 tokens)
        _layer("sdxl_1k_attn_out", 2048, 1280, 1280, "fp16"),
        # SDXL 4K stage with routed tokens (8192 and 10 odd ones), feed-forward up-projection, group-32 weights
        _layer("sdxl_routed_ff_g32", 8202, 640, 5120, "fp16", group=32),
        # SDXL 4K stage, 1280-channel block, group-32 weights, bf16 activations as the benchmark states them
        _layer("sdxl_4k_ff_g32", 16384, 1280, 5120, "bf16", group=32),
        # FLUX text stream (512 prompt tokens) through its MLP down-projection: few rows, a long K
        _layer("flux_text_mlp_down", 512, 12288, 3072, rank=32),
        # FLUX 1K stage, attention projection with the SVDQuant low-rank branch
        _layer("flux_1k_attn", 4096, 3072, 3072, rank=32),
        # FLUX 1K stage with its 256 text tokens, MLP up-projection, plain INT8
        _layer("flux_1k_mlp_up", 4352, 3072, 12288),
        # FLUX 1K stage, single-block proj_out split along its input, both halves with a low-rank branch
        {"name": "flux_1k_split_out", "kind": "split", "M": 4352, "N": 3072, "dtype": "bf16", "rank": 32},
        # FLUX 4K stage, MLP up-projection: the headline layer
        _layer("flux_4k_mlp_up", 65536, 3072, 12288, rank=32),
        # FLUX 4K stage, MLP down-projection: the same operations with a long K
        _layer("flux_4k_mlp_down", 65536, 12288, 3072, rank=32),
        # FLUX 4K stage routed: 33,316 active rows gathered, results scattered into the 65,536-row canvas
        {"name": "flux_4k_routed", "kind": "routed", "K": 3072, "N": 12288, "dtype": "bf16", "rank": 32,
         "active": 0.35, "mask_seed": 42},
        # loading a model: one FLUX MLP weight converted to INT8
        {"name": "convert_flux_mlp", "kind": "convert", "K": 3072, "N": 12288, "dtype": "bf16", "group": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


FLUX_SHAPES = sorted(FLUX_TOKEN_SHAPES) + [(3072, 9216)]   # and the fused QKV


def draw(rng):
    kind = rng.choice(["sdxl", "sdxl", "flux", "flux", "flux", "split", "routed", "convert"])
    if kind == "sdxl":
        K, N = rng.choice(SDXL_TOKEN_SHAPES)
        M = _log_int(rng, 77, 65556)
        return {"kind": "layer", "M": M, "K": K, "N": N, "dtype": rng.choice(["fp16", "fp16", "bf16"]), "rank": 0,
                "group": rng.choice([0, 32]), "bias": rng.random() < 0.7}
    if kind == "flux":
        K, N = rng.choice(FLUX_SHAPES)
        M = min(_log_int(rng, 256, 65792), MOST // (K * N))
        return {"kind": "layer", "M": M, "K": K, "N": N, "dtype": "bf16", "rank": rng.choice([0, 32, 32]), "group": 0,
                "bias": True}
    if kind == "split":
        return {"kind": "split", "M": _log_int(rng, 512, 33744), "N": 3072, "dtype": "bf16",
                "rank": rng.choice([0, 32, 32])}
    if kind == "routed":
        K, N = rng.choice([s for s in FLUX_SHAPES if s[0] == 3072])
        return {"kind": "routed", "K": K, "N": N, "dtype": "bf16", "rank": rng.choice([0, 32]),
                "active": round(rng.uniform(0.03, 0.7), 3), "mask_seed": rng.randrange(1 << 16)}
    K, N = rng.choice(FLUX_SHAPES + SDXL_TOKEN_SHAPES)
    return {"kind": "convert", "K": K, "N": N, "dtype": rng.choice(["bf16", "fp16"]), "group": rng.choice([0, 32])}


# ------------------------------------------------------------------------------------------------ inputs
def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _activations(M, K, dtype, g):
    x = torch.randn(M, K, generator=g, device=g.device)
    cols = torch.randperm(K, generator=g, device=g.device)[: max(1, round(0.005 * K))]
    x[:, cols] *= 20.0
    return x.to(dtype)


def _weights(K, N, dtype, rank, bias, g):
    """The 16-bit weight [N, K], bias [N] or None, and low-rank factors A [K, rank], B [rank, N] or None."""
    def normal(*shape, std):
        return (torch.randn(*shape, generator=g, device=g.device) * std).to(dtype)

    w = normal(N, K, std=0.02)
    b = normal(N, std=0.01) if bias else None
    ab = (normal(K, rank, std=0.02), normal(rank, N, std=0.02)) if rank else None
    return w, b, ab


def _tensors(case, seed):
    """Everything prepare() and exact() both need, from the seed alone. Each half of a split layer has its own
    low-rank factors; the bias belongs to the second."""
    g = torch.Generator(device=_dev()).manual_seed(seed)
    dt, kind = DTYPES[case["dtype"]], case["kind"]
    if kind == "split":
        K = SPLIT_AT + 12288
        x = _activations(case["M"], K, dt, g)
        w, b, _ = _weights(K, case["N"], dt, 0, True, g)
        halves = []
        for lo, hi in ((0, SPLIT_AT), (SPLIT_AT, K)):
            _, _, ab = _weights(hi - lo, case["N"], dt, case["rank"], False, g)
            halves.append((lo, hi, ab))
        return {"x": x, "w": w, "b": b, "halves": halves}
    w, b, ab = _weights(case["K"], case["N"], dt, case.get("rank", 0), case.get("bias", True), g)
    t = {"w": w, "b": b, "ab": ab}
    if kind == "layer":
        t["x"] = _activations(case["M"], case["K"], dt, g)
    elif kind == "routed":
        t["x"] = _activations(GRID * GRID, case["K"], dt, g)
        t["canvas"] = torch.randn(GRID * GRID, case["N"], generator=g, device=g.device, dtype=dt)
    return t


def _linear(w, b, ab):
    lin = nn.Linear(w.shape[1], w.shape[0], bias=b is not None, device="meta")
    lin.weight = nn.Parameter(w, requires_grad=False)
    if b is not None:
        lin.bias = nn.Parameter(b, requires_grad=False)
    if ab is not None:
        setattr(lin, LOWRANK_A_ATTR, ab[0])
        setattr(lin, LOWRANK_B_ATTR, ab[1])
    return lin


def _mask(case):
    return leaf_mask(GRID // 16, case["active"], case["mask_seed"])


def _active_rows(case):
    """The routed rows in plain torch: the active 16 x 16-token leaves, each grown by 2 tokens and clamped."""
    sel = _mask(case)
    hit = torch.zeros(GRID, GRID, dtype=torch.bool)
    for i, j in sel.nonzero().tolist():
        hit[max(0, 16 * i - 2): 16 * i + 18, max(0, 16 * j - 2): 16 * j + 18] = True
    return hit.reshape(-1).nonzero().reshape(-1)


def prepare(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    if kind == "convert":
        return {"kind": kind, "lin": _linear(t["w"], t["b"], None), "group": case["group"]}
    if kind == "split":
        K = t["w"].shape[1]
        holder = nn.Module()
        holder.proj_out = SplitInLinear(_linear(t["w"], t["b"], None), SPLIT_AT)
        for part, (_, _, ab) in zip(holder.proj_out.linears, t["halves"]):
            if ab is not None:
                setattr(part, LOWRANK_A_ATTR, ab[0])
                setattr(part, LOWRANK_B_ATTR, ab[1])
        convert_linears_to_int8(holder, whitelist=lambda name: False)
        assert holder.proj_out.in_features == K
        return {"kind": kind, "layer": holder.proj_out, "x": t["x"]}
    lin = _linear(t["w"], t["b"], t["ab"])
    if kind == "routed":
        rows = routed_row_index(_mask(case))
        return {"kind": kind, "layer": Int8Linear(lin), "x": t["x"], "rows": rows, "canvas": t["canvas"]}
    cls = SdxlInt8Linear if case["dtype"] == "fp16" or case["group"] else Int8Linear
    return {"kind": kind, "layer": cls(lin, group_size=case["group"]), "x": t["x"]}


# -------------------------------------------------------------------------------------------------- a pass
def run(state):
    if state["kind"] == "convert":
        q = Int8Linear(state["lin"], group_size=state["group"])
        return {"codes": q.weight_int8, "scale": q.w_scale, "packed": q.weight_packed, "bias": q.bias}
    if state["kind"] == "routed":
        return state["layer"](state["x"], row_idx=state["rows"], out=state["canvas"], out_row_idx=state["rows"])
    return state["layer"](state["x"])


# --------------------------------------------------------------------------------------------- what it costs
def _layer_work(M, K, N, rank, group, bias):
    scales = N * (K // group if group else 1)
    low_rank = rank * (K + N)
    return (2 * M * K + N * K + 4 * scales + (4 * N if bias else 0) + 2 * low_rank + 2 * M * N,
            2 * M * N * K + 2 * M * low_rank)


def work(case):
    kind, N = case["kind"], case["N"]
    if kind == "convert":
        K = case["K"]
        scales = N * (K // case["group"] if case["group"] else 1)
        # the 16-bit weight read once; row-major codes, kernel-layout codes, scales and the fp32 bias written once
        return {"bytes": 2 * N * K + 2 * N * K + 4 * scales + 6 * N, "flops": 4 * N * K}
    if kind == "split":
        M, parts = case["M"], (SPLIT_AT, 12288)
        b = [_layer_work(M, K, N, case["rank"], 0, False) for K in parts]
        return {"bytes": sum(v[0] for v in b) - 2 * M * N + 4 * N, "flops": sum(v[1] for v in b)}
    if kind == "routed":
        M = int(_active_rows(case).numel())
        b, f = _layer_work(M, case["K"], N, case["rank"], 0, True)
        return {"bytes": b + 8 * M, "flops": f}   # the row list, for the gather and for the scatter
    b, f = _layer_work(case["M"], case["K"], N, case["rank"], case["group"], case["bias"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Measured against exact(): 1.6e-3 to 1.9e-3 in bf16 and 2.6e-4 to 3.8e-4 in fp16 for a single layer (the rounding of
    the outputs, and of t where there is a low-rank branch), 2.6e-3 for a split one (the first half is rounded too).
    Four times that. Conversion yields the same codes, layout and scales, bit for bit."""
    if case["kind"] == "convert":
        return "exact"
    if case["dtype"] == "fp16":
        return {"rel": 1.5e-3}
    return {"rel": 1e-2 if case["kind"] == "split" else 7e-3}


# ------------------------------------------------------------------------------------------- in 64 bits
def _rtn(v):
    """Per-row round to nearest of v [..., n] (the scale is an fp32 number by definition): codes, scales."""
    v = v.double()
    s = (v.abs().amax(-1, keepdim=True).clamp_min(1e-8).float() / 127.0).double()
    return (v / s).round().clamp(-127, 127), s


def _exact_linear(x, w, ab, group, bias):
    N, K = w.shape
    qw, sw = _rtn(w.reshape(N, K // group, group) if group else w)
    wd = (qw * sw).reshape(N, K)
    out = torch.empty(x.shape[0], N, dtype=torch.float64, device=x.device)
    for r in range(0, x.shape[0], 8192):
        xr = x[r: r + 8192]
        q, s = _rtn(xr)
        y = (q @ wd.t()) * s
        if ab is not None:
            y += (xr.double() @ ab[0].double()) @ ab[1].double()
        if bias is not None:
            y += bias.double()
        out[r: r + 8192] = y
    return out


def exact(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    if kind == "convert":
        w = t["w"]
        g = case["group"] or w.shape[1]
        _, s = _rtn(w.reshape(w.shape[0], -1, g))
        return {"codes": None, "scale": s[..., 0] if case["group"] else s[:, 0, 0], "packed": None,
                "bias": t["b"].double()}
    if kind == "split":
        parts = [_exact_linear(t["x"][:, lo:hi], t["w"][:, lo:hi], ab, 0, t["b"] if lo else None)
                 for lo, hi, ab in t["halves"]]
        return parts[0] + parts[1]
    if kind == "routed":
        rows = _active_rows(case).to(t["x"].device)
        out = t["canvas"].double()
        out[rows] = _exact_linear(t["x"][rows], t["w"], t["ab"], 0, t["b"])
        return out
    return _exact_linear(t["x"], t["w"], t["ab"], case["group"], t["b"])
