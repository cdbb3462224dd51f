"""The work that users of piper_offload_amd have it do, as cases to be timed and compared.

A LoRA merge library is called for whole models (grouped merges of every projection), for single weights of every
storage format, for the two halves of the portable path (decode a weight to dense, encode a dense weight) and for the
routed residual that stands in for a merge at inference.  Sizes are those of the repository's benchmark (the projections
of an 8B-shaped model, the single-weight configurations) and generic Linear shapes around them.

``listed()`` names one case for each of these, ``draw()`` gives more over the same ranges.  A case is a dict of plain
values:

* ``op``: stack | merge | dequant | requant | routed
* ``fmt``: int8 | fp8 | nvfp4 | mxfp4 | mxfp8 | q8_0 | dense, or a GGUF type for ``dequant``
* ``rows``, ``cols`` (the weight is [out, in] = [rows, cols]), ``rank``, ``tokens``, ``layers``
* ``layout``: row | tensor | group (qparams of int8 / fp8; groups of 128), plain | swizzled (block scales)
* ``sr``: stochastic rounding; ``dtype``: the compute dtype; ``asym``: INT8 with zero points
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "piper-offload_amd"))

from piper_offload_amd import Int8Weight, NVFP4Weight, derive_seed  # noqa: E402
from piper_offload_amd import kernels as K  # noqa: E402
from piper_offload_amd.routed import RoutedFactor, routed_residual  # noqa: E402
from piper_offload_amd.stack import StackPlan, StackTarget  # noqa: E402

# the projections of one layer of the 8B-shaped model of bench.py
LAYER = (("q", 4096, 4096), ("k", 1024, 4096), ("v", 1024, 4096), ("o", 4096, 4096),
         ("gate", 14336, 4096), ("up", 14336, 4096), ("down", 4096, 14336))
GROUP = 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
GGUF = {"f16": (1, 1, 2), "bf16": (30, 1, 2), "q4_0": (2, 32, 18), "q8_0": (8, 32, 34), "q4_k": (12, 256, 144),
        "q5_k": (13, 256, 176), "q6_k": (14, 256, 210)}  # type id, elements and bytes per block
MX_ELEM = {"mxfp4": torch.float4_e2m1fn_x2, "mxfp8": torch.float8_e4m3fn}


def listed():
    return [
        # the smallest call: one small projection, where the launches and the host side count
        dict(name="int8 small merge", op="merge", fmt="int8", rows=320, cols=768, rank=8, layout="row", sr=False,
             dtype="bf16", asym=False),
        # a whole model merged once: every projection of the 8B-shaped INT8 model in one grouped merge (bench.py's default)
        dict(name="int8 8B stack", op="stack", fmt="int8", layers=32, rank=16, layout="row", sr=True),
        # merge on reload: one layer of the NVFP4 model as a block is loaded
        dict(name="nvfp4 layer stack", op="stack", fmt="nvfp4", layers=1, rank=16, layout="plain", sr=False),
        # the single-weight configurations of the benchmark: scaled FP8 per row at a high rank
        dict(name="fp8 row merge r64", op="merge", fmt="fp8", rows=8192, cols=8192, rank=64, layout="row", sr=True,
             dtype="bf16"),
        # scaled-FP8 checkpoints with one scale per tensor, ragged rows
        dict(name="fp8 tensor merge", op="merge", fmt="fp8", rows=13800, cols=5120, rank=32, layout="tensor", sr=False,
             dtype="bf16"),
        # GGUF Q8_0, the benchmark's configuration
        dict(name="q8_0 merge", op="merge", fmt="q8_0", rows=13824, cols=5120, rank=16, sr=False, dtype="bf16"),
        # MXFP8 weights, scales in the swizzled order that matmul kernels want
        dict(name="mxfp8 merge", op="merge", fmt="mxfp8", rows=14336, cols=4096, rank=16, layout="swizzled", sr=True,
             dtype="bf16"),
        # plain bf16 weights, the most usual merge of all
        dict(name="dense merge", op="merge", fmt="dense", rows=4096, cols=14336, rank=32, dtype="bf16"),
        # decode: a packed weight to dense values (the portable path's first half, and inference without packed matmuls)
        dict(name="nvfp4 dequant", op="dequant", fmt="nvfp4", rows=14336, cols=4096, layout="plain", dtype="bf16"),
        # encode: a dense weight to a packed format
        dict(name="int8 requant", op="requant", fmt="int8", rows=4096, cols=4096, layout="row", sr=False, dtype="bf16",
             asym=False),
        # routed LoRA: decode and prefill
        dict(name="routed decode", op="routed", fmt="dense", tokens=1, rows=14336, cols=4096, rank=16, dtype="bf16"),
        dict(name="routed prefill", op="routed", fmt="dense", tokens=4096, rows=14336, cols=4096, rank=16, dtype="bf16"),
    ]


def _spread(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, unit):
    return max(unit, int(_spread(rng, lo, hi)) // unit * unit)


def draw(rng: random.Random):
    op = rng.choice(["merge"] * 5 + ["dequant", "dequant", "requant", "requant", "routed", "routed", "stack"])
    rank = rng.choice([4, 8, 16, 16, 24, 32, 64])
    sr = rng.random() < 0.5
    if op == "stack":
        fmt = rng.choice(["int8", "nvfp4"])
        return dict(op=op, fmt=fmt, layers=rng.randint(1, 8), rank=rng.choice([8, 16, 16, 32]),
                    layout="row" if fmt == "int8" else rng.choice(["plain", "swizzled"]), sr=sr)
    if op == "routed":
        t = _size(rng, 1, 8192, 1)
        n = _size(rng, 256, 16384, rng.choice([8, 64, 128]))
        return dict(op=op, fmt="dense", tokens=t, rows=min(n, max(256, (1 << 27) // t // 8 * 8)),
                    cols=_size(rng, 256, 16384, rng.choice([8, 64, 128])), rank=rank, dtype=rng.choice(["bf16", "bf16", "f16"]))
    fmts = {"merge": ["int8", "int8", "fp8", "fp8", "nvfp4", "mxfp4", "mxfp8", "q8_0", "dense", "dense"],
            "dequant": ["int8", "fp8", "nvfp4", "mxfp4", "mxfp8"] + sorted(GGUF),
            "requant": ["int8", "fp8", "nvfp4", "mxfp4", "mxfp8", "q8_0"]}[op]
    fmt = rng.choice(fmts)
    layout = {"int8": ["row", "row", "group", "tensor"], "fp8": ["row", "tensor", "group"],
              "nvfp4": ["plain", "swizzled"], "mxfp4": ["plain", "swizzled"], "mxfp8": ["plain", "swizzled"]}.get(fmt)
    layout = rng.choice(layout) if layout else None
    # columns: what the format's blocks allow, mostly the multiples of 64 or 128 that models have, sometimes less even
    least = {"nvfp4": 16, "mxfp4": 32, "mxfp8": 32, "q8_0": 32}.get(fmt, 1)
    if fmt in GGUF and op == "dequant":
        least = max(GGUF[fmt][1], 8)
    unit = rng.choice([128, 128, 64, max(least, 8), least])
    if layout == "group":
        unit = GROUP
    unit = max(unit, least)
    rows, cols = _size(rng, 64, 16384, rng.choice([1, 16, 128])), _size(rng, max(256, 2 * unit), 16384, unit)
    rows = min(rows, (1 << 27) // cols)
    case = dict(op=op, fmt=fmt, rows=rows, cols=cols, dtype=rng.choice(["bf16", "bf16", "bf16", "f16"]))
    if fmt in ("nvfp4", "mxfp4", "mxfp8") and op != "dequant" or fmt == "q8_0":
        case["dtype"] = "bf16"  # the compute dtype of these formats
    if op == "merge":
        case["rank"] = rank
    if op != "dequant" and fmt != "dense":
        case["sr"] = sr
    if layout:
        case["layout"] = layout
    if fmt == "int8":
        case["asym"] = rng.random() < 0.25
    return case


# ---------------------------------------------------------------------------
# inputs, in plain torch: weights ~ N(0, 0.02), A ~ N(0, 1/rank), B ~ N(0, 0.01)
# ---------------------------------------------------------------------------
def _normal(g, shape, std, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _factors(g, rows, cols, rank, dtype=torch.bfloat16):
    return _normal(g, (rows, rank), 0.01, dtype), _normal(g, (rank, cols), 1.0 / rank, dtype)


def _block_size(case):
    rows, cols = case["rows"], case["cols"]
    return {"row": (1, cols), "tensor": (rows, cols), "group": (1, GROUP)}[case["layout"]]


def _grouped(case, t):
    """[rows, cols] as [qparams, elements of each]."""
    r, c = _block_size(case)
    return t.reshape(-1, r * c)


def _qshape(case):
    r, c = _block_size(case)
    return (case["rows"] // r, case["cols"] // c)


def _int8_encode(w, asym):
    """w [n, k] float: codes, scale [n, 1], zero point [n, 1] or None."""
    if asym:
        mx, mn = w.amax(1, keepdim=True).clamp_min(0), w.amin(1, keepdim=True).clamp_max(0)
        s = ((mx - mn) / 255).clamp_min(1e-7)
        z = (-128 - torch.round(mn / s)).clamp(-128, 127)
        return torch.round(w / s + z).clamp_(-128, 127).to(torch.int8), s, z.to(torch.int8)
    s = (w.abs().amax(1, keepdim=True) / 127).clamp_min(1e-7)
    return torch.round(w / s).clamp_(-128, 127).to(torch.int8), s, None


_FP4_MID = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)
_FP4_VAL = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _fp4_pack(x):
    """Nearest e2m1 codes of x, two to a byte, the even column in the low nibble."""
    mid = torch.tensor(_FP4_MID, device=x.device)
    code = torch.bucketize(x.abs(), mid, out_int32=True).to(torch.uint8) | (torch.signbit(x).to(torch.uint8) << 3)
    return (code[:, 0::2] | (code[:, 1::2] << 4)).contiguous()


def _fp4_values(packed):
    val = torch.tensor(_FP4_VAL + tuple(-v for v in _FP4_VAL), device=packed.device, dtype=torch.float64)
    return torch.stack((val[(packed & 15).long()], val[(packed >> 4).long()]), -1).reshape(packed.shape[0], -1)


def _swizzle(s):
    """Plain block scales [rows, n] as the 128 x 4 tiles of the swizzled order, zero-padded."""
    rows, n = s.shape
    rb, cb = (rows + 127) // 128, (n + 3) // 4
    pad = torch.zeros((rb * 128, cb * 4), dtype=s.dtype, device=s.device)
    pad[:rows, :n] = s
    return pad.reshape(rb, 4, 32, cb, 4).permute(0, 3, 2, 1, 4).reshape(rb * 32, cb * 16).contiguous()


def _nvfp4_encode(w):
    """w [rows, cols] float: packed codes, e4m3 block scales as bytes [rows, cols / 16], global scale."""
    rows, cols = w.shape
    blocks = w.reshape(rows, cols // 16, 16)
    pts = (w.abs().amax() / 2688).clamp_min(1e-7)
    s = (blocks.abs().amax(2) / 6 / pts).clamp(0.015625, 448).to(torch.float8_e4m3fn)
    q = _fp4_pack((blocks / (s.float() * pts).unsqueeze(2)).reshape(rows, cols))
    return q, s.view(torch.uint8), pts


def _mx_encode(w, fmt):
    """w [rows, cols] float: codes (packed bytes or fp8) and e8m0 scales as bytes, floor mode."""
    rows, cols = w.shape
    blocks = w.reshape(rows, cols // 32, 32)
    e = torch.floor(torch.log2(blocks.abs().amax(2).clamp_min(2.0**-100))) - (2 if fmt == "mxfp4" else 8)
    x = (blocks * torch.exp2(-e).unsqueeze(2)).reshape(rows, cols)
    q = _fp4_pack(x.clamp_(-6, 6)) if fmt == "mxfp4" else x.clamp_(-448, 448).to(torch.float8_e4m3fn)
    return q, (e + 127).to(torch.uint8)


def _gguf_bytes(g, fmt, rows, cols):
    """Random blocks of one type: codes of every value, scales as the encoders give them."""
    _, block, nbytes = GGUF[fmt]
    if block == 1:
        return _normal(g, (rows, cols), 0.02, DTYPES[fmt]).view(torch.uint8)
    n = rows * cols // block
    raw = torch.randint(0, 256, (n, nbytes), generator=g, device="cuda", dtype=torch.uint8)
    for off in {"q4_0": (0,), "q8_0": (0,), "q4_k": (0, 2), "q5_k": (0, 2), "q6_k": (208,)}[fmt]:
        d = torch.rand((n, 1), generator=g, device="cuda").mul_(9e-4).add_(1e-4).to(torch.float16)
        raw[:, off:off + 2] = d.view(torch.uint8)
    return raw.reshape(rows, -1)


def _inputs(case, seed):
    """Everything a case starts from, as plain tensors made from the seed."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = {}
    if case["op"] == "stack":
        return d
    rows, cols, op, fmt = case["rows"], case["cols"], case["op"], case["fmt"]
    dt = DTYPES[case["dtype"]]
    if op == "routed":
        d["x"], d["y"] = _normal(g, (case["tokens"], cols), 1.0, dt), _normal(g, (case["tokens"], rows), 1.0, dt)
        d["b"], d["a"] = _factors(g, rows, cols, case["rank"], dt)
        return d
    if fmt in GGUF and (op == "dequant" or fmt == "q8_0" and op == "merge"):
        if op == "merge":
            w = _normal(g, (rows, cols), 0.02).float().reshape(-1, 32)
            s = w.abs().amax(1, keepdim=True) / 127
            q = torch.round(w / s.clamp_min(1e-7)).clamp_(-127, 127).to(torch.int8)
            raw = torch.cat((s.to(torch.float16).view(torch.uint8), q.view(torch.uint8)), 1)
            d["q"] = raw.reshape(rows, -1)
        else:
            d["q"] = _gguf_bytes(g, fmt, rows, cols)
    elif op == "requant" or fmt == "dense":
        d["w"] = _normal(g, (rows, cols), 0.02, dt)
    else:
        w = _normal(g, (rows, cols), 0.02).float()
        if fmt == "int8":
            q, d["s"], d["z"] = _int8_encode(_grouped(case, w), case["asym"])
            d["q"], d["s"] = q.reshape(rows, cols), d["s"].reshape(_qshape(case))
            d["z"] = None if d["z"] is None else d["z"].reshape(_qshape(case))
        elif fmt == "fp8":
            wg = _grouped(case, w)
            s = (wg.abs().amax(1, keepdim=True) / 448).clamp_min(1e-7)
            d["q"] = (wg / s).clamp_(-448, 448).to(torch.float8_e4m3fn).reshape(rows, cols)
            d["s"] = s.reshape(_qshape(case))
        elif fmt == "nvfp4":
            d["q"], d["s"], d["pts"] = _nvfp4_encode(w)
        else:
            d["q"], d["s"] = _mx_encode(w, fmt)
        del w
    if op == "merge":
        d["b"], d["a"] = _factors(g, rows, cols, case["rank"], dt)
    return d


def _stack_shapes(case):
    return [(f"layers.{i}.{name}.weight", r, c) for i in range(case["layers"]) for name, r, c in LAYER]


def _stack_inputs(case, seed):
    """(path, rows, cols, generator) of every target, each with inputs of its own."""
    for i, (path, r, c) in enumerate(_stack_shapes(case)):
        yield path, r, c, torch.Generator(device="cuda").manual_seed(seed * 1009 + i)


def prepare(case, seed):
    if case["op"] != "stack":
        d = _inputs(case, seed)
        if case.get("layout") == "swizzled" and "s" in d:
            d["s"] = _swizzle(d["s"])
        if case["fmt"] == "nvfp4" and "s" in d:
            d["s"] = d["s"].view(torch.float8_e4m3fn)
        if case["op"] == "routed":
            d["factors"] = [RoutedFactor(d["a"], d["b"], 1.0)]
        d["case"], d["seed"] = case, derive_seed("layers.0.proj.weight", seed) if case.get("sr") else None
        return d
    # the targets' storage lies in one buffer for codes and one for scales, as a loader of whole checkpoints lays it out
    shapes = _stack_shapes(case)
    total = sum(r * c for _, r, c in shapes)
    swz = case["layout"] == "swizzled"
    if case["fmt"] == "int8":
        codes = torch.empty(total, dtype=torch.int8, device="cuda")
        scales = torch.empty(sum(r for _, r, _c in shapes), device="cuda")
        out = {"codes": codes, "scales": scales}
    else:
        codes = torch.empty(total // 2, dtype=torch.uint8, device="cuda")
        scales = torch.empty(total // 16, dtype=torch.uint8, device="cuda")
        out = {"codes": codes, "scales": scales, "pts": torch.empty(len(shapes), device="cuda")}
    targets, at, at_s = [], 0, 0
    for i, (path, r, c, g) in enumerate(_stack_inputs(case, seed)):
        w = _normal(g, (r, c), 0.02).float()
        if case["fmt"] == "int8":
            q, s, _ = _int8_encode(w, False)
            qv, sv = codes[at:at + r * c].view(r, c), scales[at_s:at_s + r].view(r, 1)
            weight = Int8Weight(qv, sv, (1, c), torch.bfloat16)
        else:
            q, s, p = _nvfp4_encode(w)
            s = _swizzle(s) if swz else s
            qv, sv = codes[at:at + q.numel()].view(q.shape), scales[at_s:at_s + s.numel()].view(s.shape)
            out["pts"][i] = p
            weight = NVFP4Weight(qv, sv.view(torch.float8_e4m3fn), out["pts"][i], 16, is_swizzled_scales=swz)
        qv.copy_(q)
        sv.copy_(s)
        at, at_s = at + q.numel(), at_s + s.numel()
        b, a = _factors(g, r, c, case["rank"])
        targets.append(StackTarget(weight, b, a, 1.0, derive_seed(path, seed)))
        del w, q, s
    return {"case": case, "plan": StackPlan(targets, case["fmt"]), "seeds": [t.seed for t in targets], "out": out}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _u8(t):
    return t.view(torch.uint8)


def run(state):
    case = state["case"]
    op, fmt = case["op"], case["fmt"]
    if op == "stack":
        state["plan"].merge(state["seeds"], stochastic=case["sr"])
        return state["out"]
    if op == "routed":
        return routed_residual(state["x"], state["factors"], state["y"])
    if op == "merge":
        return _merge(state, case, fmt)
    if op == "dequant":
        return _dequant(state, case, fmt)
    return _requant(state, case, fmt)


def _merge(st, case, fmt):
    b, a, seed = st["b"], st["a"], st["seed"]
    if fmt == "dense":
        K.merge_dense_lora_(st["w"], b, a, 1.0)
        return st["w"]
    if fmt == "int8":
        q, s, z = K.merge_int8_lora(st["q"], st["s"], st["z"], _block_size(case), b, a, 1.0, asymmetric=case["asym"],
                                    reduce_range=False, rounding_seed=seed)
        return {"q": q, "s": s, "z": z}
    if fmt == "fp8":
        q, s = K.merge_float8_lora(st["q"], st["s"], _block_size(case), b, a, 1.0, rounding_seed=seed)
        return {"q": _u8(q), "s": s}
    if fmt == "nvfp4":
        q, s, p = K.merge_nvfp4_lora(st["q"], st["s"], st["pts"], 16, case["layout"] == "swizzled", b, a, 1.0,
                                     rounding_seed=seed)
        return {"q": q, "s": _u8(s), "pts": p}
    if fmt == "q8_0":
        return K.merge_q8_0_lora(st["q"], b, a, 1.0, rounding_seed=seed)
    K.merge_mx_lora_(st["q"], st["s"], MX_ELEM[fmt], 32, torch.bfloat16, b, a, 1.0, scaling_mode=0,
                     swizzled=case["layout"] == "swizzled", rounding_seed=seed)
    return {"q": _u8(st["q"]), "s": st["s"]}


def _dequant(st, case, fmt):
    dt = DTYPES[case["dtype"]]
    if fmt in GGUF:
        return K.dequantize_gguf(st["q"], GGUF[fmt][0], dtype=dt)
    if fmt == "int8":
        return K.dequantize_int8(st["q"], st["s"], st["z"], _block_size(case), dtype=dt)
    if fmt == "fp8":
        return K.dequantize_float8(st["q"], st["s"], _block_size(case), dtype=dt)
    swz = case["layout"] == "swizzled"
    if fmt == "nvfp4":
        return K.dequantize_nvfp4(st["q"], st["s"], st["pts"], swizzled=swz, dtype=dt)
    return K.dequantize_mx(st["q"], st["s"], MX_ELEM[fmt], case["cols"], swizzled=swz, dtype=dt)


def _requant(st, case, fmt):
    w, seed = st["w"], st["seed"]
    if fmt == "int8":
        q, s, z = K.requantize_int8(w, _block_size(case), asymmetric=case["asym"], rounding_seed=seed)
        return {"q": q, "s": s, "z": z}
    if fmt == "fp8":
        q, s = K.requantize_float8(w, _block_size(case), rounding_seed=seed)
        return {"q": _u8(q), "s": s}
    if fmt == "q8_0":
        return K.requantize_q8_0(w, rounding_seed=seed)
    swz = case["layout"] == "swizzled"
    if fmt == "nvfp4":
        q, s, p = K.requantize_nvfp4(w, two_level=True, swizzled=swz, rounding_seed=seed)
        return {"q": q, "s": _u8(s), "pts": p}
    q, s = K.requantize_mx(w, MX_ELEM[fmt], swizzled=swz, rounding_seed=seed)
    return {"q": _u8(q), "s": s}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close another implementation comes
# ---------------------------------------------------------------------------
def _stored_bytes(case, rows, cols):
    """Bytes of one stored weight, codes and qparams."""
    n, fmt = rows * cols, case["fmt"]
    if fmt in ("int8", "fp8"):
        q = {"row": rows, "tensor": 1, "group": n // GROUP}[case["layout"]]
        return n + q * (5 if case.get("asym") else 4)
    if fmt in GGUF:
        return n // GGUF[fmt][1] * GGUF[fmt][2]
    return {"nvfp4": n // 2 + n // 16 + 4, "mxfp4": n // 2 + n // 32, "mxfp8": n + n // 32, "dense": 2 * n}[fmt]


def work(case):
    if case["op"] == "stack":
        shapes, r = [(m, n) for _, m, n in LAYER], case["rank"]
        return {"bytes": case["layers"] * sum(2 * _stored_bytes(case, m, n) + 2 * r * (m + n) for m, n in shapes),
                "flops": case["layers"] * sum(2 * r * m * n for m, n in shapes)}
    m, n, r = case["rows"], case["cols"], case.get("rank", 0)
    if case["op"] == "routed":
        t = case["tokens"]
        return {"bytes": 2 * (t * n + 2 * t * m + r * (m + n)), "flops": 2 * t * r * (m + n)}
    stored = _stored_bytes(case, m, n)
    if case["op"] == "merge":
        return {"bytes": 2 * stored + 2 * r * (m + n), "flops": 2 * r * m * n}
    return {"bytes": stored + 2 * m * n, "flops": 0}


def tolerance(case):
    # Codes, scales and decoded values are determined to the bit by the formats' recipes: the merged value's fp32 delta
    # is rounded to the compute dtype before it is encoded.  Dense results carry the order of the 32-bit sums into the
    # last bit of a few of their 16-bit values (one ulp is 2^-8 of a bf16 value): sums taken in another order differed
    # by rel 1.6e-5 and max 0.0077 at most (routed) and 3e-6 and 0.0076 (dense merge), and one value in a result of 256
    # makes rel 2.4e-4 by itself.
    if case["op"] == "routed":
        return {"rel": 5e-4, "max": 0.031}
    if case["op"] == "merge" and case["fmt"] == "dense":
        return {"rel": 1e-4, "max": 0.031}
    return "exact"


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _delta(d):
    return d["b"].double() @ d["a"].double()


def _stored_values(case, d):
    """The dequantized weight in 64 bits."""
    fmt = case["fmt"]
    if fmt in ("int8", "fp8"):
        q = d["q"].double()
        x = _grouped(case, q)
        z = d.get("z")
        if z is not None:
            x = x - z.double().reshape(-1, 1)
        return (x * d["s"].double().reshape(-1, 1)).reshape(q.shape)
    if fmt == "nvfp4":
        s = d["s"].view(torch.float8_e4m3fn).double() * d["pts"].double()
        return _fp4_values(d["q"]) * s.repeat_interleave(16, 1)
    if fmt in ("mxfp4", "mxfp8"):
        x = _fp4_values(d["q"]) if fmt == "mxfp4" else d["q"].double()
        return x * torch.exp2(d["s"].double() - 127).repeat_interleave(32, 1)
    return _gguf_values(fmt, d["q"], case["cols"])


def _f16(raw):
    return raw.contiguous().view(torch.float16).double()


def _gguf_values(fmt, raw, cols):
    """GGUF blocks by their published layouts."""
    rows = raw.shape[0]
    if GGUF[fmt][1] == 1:
        return raw.view(DTYPES[fmt]).double()
    b = raw.reshape(-1, GGUF[fmt][2])
    n = b.shape[0]
    if fmt == "q8_0":
        return (_f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if fmt == "q4_0":
        q = torch.cat((b[:, 2:] & 15, b[:, 2:] >> 4), 1).double() - 8
        return (_f16(b[:, :2]) * q).reshape(rows, cols)
    if fmt in ("q4_k", "q5_k"):
        d, dmin, sc = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16]
        s = torch.cat((sc[:, 0:4] & 63, (sc[:, 8:12] & 15) | ((sc[:, 0:4] >> 6) << 4)), 1).double()
        m = torch.cat((sc[:, 4:8] & 63, (sc[:, 8:12] >> 4) | ((sc[:, 4:8] >> 6) << 4)), 1).double()
        qs = b[:, 16 if fmt == "q4_k" else 48:].reshape(n, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).reshape(n, 8, 32).to(torch.int64)
        if fmt == "q5_k":
            bit = torch.arange(8, device=b.device).reshape(1, 8, 1)
            q = q + (((b[:, 16:48].to(torch.int64).unsqueeze(1) >> bit) & 1) << 4)
        return ((d * s).unsqueeze(2) * q.double() - (dmin * m).unsqueeze(2)).reshape(rows, cols)
    # q6_k
    ql, qh = b[:, :128].reshape(n, 2, 2, 32).to(torch.int64), b[:, 128:192].reshape(n, 2, 1, 32).to(torch.int64)
    lo = torch.stack((ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4), 2)
    hi = (qh >> torch.tensor([0, 2, 4, 6], device=b.device).reshape(1, 1, 4, 1)) & 3
    q = (lo | (hi << 4)).double().sub(32).reshape(n, 16, 16)
    s = b[:, 192:208].contiguous().view(torch.int8).double()
    return (_f16(b[:, 208:210]) * s).unsqueeze(2).mul(q).reshape(rows, cols)


def _exact_encoded(case, m):
    """The outputs of an encode of m: the scales that are floating numbers; codes and packed scales have no 64-bit value."""
    fmt = case["fmt"]
    if fmt in ("int8", "fp8"):
        x = _grouped(case, m)
        if fmt == "fp8":
            return {"q": None, "s": (x.abs().amax(1) / 448).reshape(_qshape(case))}
        if case["asym"]:
            s = (x.amax(1).clamp_min(0) - x.amin(1).clamp_max(0)) / 255
        else:
            s = x.abs().amax(1) / 127.5
        return {"q": None, "s": s.reshape(_qshape(case)), "z": None}
    if fmt == "nvfp4":
        return {"q": None, "s": None, "pts": m.abs().amax() / 2688}
    return None  # bytes only


def exact(case, seed):
    op, fmt = case["op"], case["fmt"]
    if op == "stack":
        got = []
        for _path, r, c, g in _stack_inputs(case, seed):
            w = _normal(g, (r, c), 0.02).float()
            one = dict(case, rows=r, cols=c, asym=False)
            d = {}
            if fmt == "int8":
                d["q"], d["s"], d["z"] = _int8_encode(w, False)
            else:
                d["q"], d["s"], d["pts"] = _nvfp4_encode(w)
            del w
            d["b"], d["a"] = _factors(g, r, c, case["rank"])
            e = _exact_encoded(one, _stored_values(one, d) + _delta(d))
            got.append((e["s"] if fmt == "int8" else e["pts"]).reshape(-1))
        return {"codes": None, "scales": torch.cat(got)} if fmt == "int8" else {"codes": None, "scales": None, "pts": torch.cat(got)}
    d = _inputs(case, seed)
    if op == "routed":
        return d["y"].double() + (d["x"].double() @ d["a"].double().T) @ d["b"].double().T
    if op == "dequant":
        return _stored_values(case, d)
    if op == "requant":
        return _exact_encoded(case, d["w"].double())
    if fmt == "dense":
        return d["w"].double() + _delta(d)
    return None if fmt == "q8_0" else _exact_encoded(case, _stored_values(case, d) + _delta(d))
