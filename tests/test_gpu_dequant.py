"""Decode of packed weights to dense values (csrc/lm_dequant.h) against the oracle, bit for bit: every code, rows of odd
length (a lane's 8 elements cross into the next row), the last elements that fill no lane, more than one workgroup,
misaligned codes, every qparam layout and output dtype."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from piper_offload_amd import kernels as K

pytestmark = pytest.mark.gpu

OUT = {torch.bfloat16: O.DT_BF16, torch.float16: O.DT_F16, torch.float32: O.DT_BF16}  # fp32 outputs hold bf16 values
FP4 = getattr(torch, "float4_e2m1fn_x2", None)


def _check(got: torch.Tensor, want_bits: np.ndarray, dtype: torch.dtype) -> None:
    want = torch.from_numpy(want_bits.view(np.int16)).view(torch.float16 if dtype is torch.float16 else torch.bfloat16)
    want = want.reshape(got.shape).to(dtype)
    got = got.cpu()
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    bits = torch.int32 if dtype is torch.float32 else torch.int16
    assert torch.equal(got.view(bits)[~nan], want.view(bits)[~nan])


def _f16_block_values(values: np.ndarray, scale: np.ndarray, block: int, swizzled: bool, g: np.ndarray | None) -> np.ndarray:
    """fp16 bits of value * scale, each step rounded to fp16 (the oracle's block formats round to bf16 only)."""
    rows, cols = values.shape
    n = cols // block
    s = np.empty((rows, n), np.float32)
    for r in range(rows):
        for c in range(n):
            s[r, c] = scale.reshape(-1)[O.blocked_scale_offset(r, c, n, swizzled)]
    with np.errstate(over="ignore", invalid="ignore"):
        s = s.astype(np.float16).astype(np.float32)
        if g is not None:
            s = (s * g).astype(np.float16).astype(np.float32)
        return (values * np.repeat(s, block, 1)).astype(np.float16).view(np.uint16)


def _fp4_values(q: np.ndarray) -> np.ndarray:
    mag = np.array([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], np.float32)
    val = np.concatenate([mag, -mag])
    return np.stack([val[q & 15], val[q >> 4]], -1).reshape(q.shape[0], -1)


def _dev(a: np.ndarray, misaligned: bool = False) -> torch.Tensor:
    t = torch.from_numpy(np.ascontiguousarray(a))
    if not misaligned:
        return t.cuda()
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    flat[1:] = t.reshape(-1).cuda()
    return flat[1:].view(t.shape)


def _group(layout: str, rows: int, cols: int) -> tuple[tuple[int, int], int]:
    return {"row": ((1, cols), cols), "tensor": ((rows, cols), rows * cols), "g16": ((1, 16), 16)}[layout]


SHAPES = [(1, 64), (3, 41), (7, 13), (65, 1003), (33, 2048)]
LAYOUTS = [(sh, lay) for sh in SHAPES for lay in ("row", "tensor", "g16") if lay != "g16" or sh[1] % 16 == 0]


@pytest.mark.parametrize("dtype", list(OUT))
@pytest.mark.parametrize("shape,layout", LAYOUTS)
def test_int8(shape: tuple[int, int], layout: str, dtype: torch.dtype) -> None:
    rows, cols = shape
    rng = np.random.default_rng(rows * cols)
    block, g = _group(layout, rows, cols)
    nq = rows * cols // g
    q = rng.integers(-128, 128, shape).astype(np.int8)
    for zp in (None, rng.integers(-128, 128, nq).astype(np.int8)):
        for sdt in (torch.float32, torch.bfloat16):
            s = torch.from_numpy(rng.normal(0, 0.01, nq).astype(np.float32)).to(sdt)
            s_or = s.numpy() if sdt is torch.float32 else s.view(torch.int16).numpy().view(np.uint16)
            want = O.int8_dequant(q, s_or, zp, g, scale_dt=O.DT_F32 if sdt is torch.float32 else O.DT_BF16, cd=OUT[dtype])
            for off in (False, True):
                got = K.dequantize_int8(_dev(q, off), s.cuda(), None if zp is None else _dev(zp), block, dtype=dtype)
                _check(got, want, dtype)


@pytest.mark.parametrize("dtype", list(OUT))
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("shape,layout", LAYOUTS)
def test_fp8(shape: tuple[int, int], fp8: torch.dtype, layout: str, dtype: torch.dtype) -> None:
    rows, cols = shape
    rng = np.random.default_rng(rows * cols + 1)
    block, g = _group(layout, rows, cols)
    q = rng.integers(0, 256, shape).astype(np.uint8)
    sshape = {"row": (rows, 1), "tensor": (1, 1), "g16": (rows, cols // 16)}[layout]
    s = rng.normal(0, 0.01, sshape).astype(np.float32)
    want = O.fp8_dequant(q, s.reshape(-1), g, fmt=O.DT_E4M3 if fp8 is torch.float8_e4m3fn else O.DT_E5M2, cd=OUT[dtype])
    for off in (False, True):
        _check(K.dequantize_float8(_dev(q, off).view(fp8), _dev(s), block, dtype=dtype), want, dtype)


BLOCK_SHAPES = [(1, 32), (5, 96), (129, 160), (33, 2080)]


@pytest.mark.parametrize("dtype", list(OUT))
@pytest.mark.parametrize("swizzled", [False, True])
@pytest.mark.parametrize("shape", BLOCK_SHAPES)
def test_nvfp4(shape: tuple[int, int], swizzled: bool, dtype: torch.dtype) -> None:
    rows, cols = shape
    rng = np.random.default_rng(rows * cols + 2)
    q = rng.integers(0, 256, (rows, cols // 2)).astype(np.uint8)
    s = rng.integers(0, 256, O.blocked_scale_shape(rows, cols, 16, swizzled)).astype(np.uint8)
    for g in (None, np.float32(0.0123)):
        if dtype is torch.float16:
            want = _f16_block_values(_fp4_values(q), O.fp8_to_f32(s), 16, swizzled, g)
        else:
            want = O.nvfp4_dequant(q, s, g, swizzled=swizzled, cd=OUT[dtype])
        gd = None if g is None else torch.tensor(float(g), device="cuda")
        for off in (False, True):
            got = K.dequantize_nvfp4(_dev(q, off), _dev(s).view(torch.float8_e4m3fn), gd, swizzled=swizzled, dtype=dtype)
            _check(got, want, dtype)


@pytest.mark.parametrize("dtype", list(OUT))
@pytest.mark.parametrize("swizzled", [False, True])
@pytest.mark.parametrize("elem", [FP4, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("shape", BLOCK_SHAPES)
def test_mx(shape: tuple[int, int], elem: torch.dtype, swizzled: bool, dtype: torch.dtype) -> None:
    rows, cols = shape
    rng = np.random.default_rng(rows * cols + 3)
    q = rng.integers(0, 256, (rows, cols // 2 if elem is FP4 else cols)).astype(np.uint8)
    s = rng.integers(0, 256, O.blocked_scale_shape(rows, cols, 32, swizzled)).astype(np.uint8)
    fmt = {FP4: O.DT_E2M1, torch.float8_e4m3fn: O.DT_E4M3, torch.float8_e5m2: O.DT_E5M2}[elem]
    if dtype is torch.float16:
        values = _fp4_values(q) if elem is FP4 else O.fp8_to_f32(q, fmt)
        want = _f16_block_values(values, O.e8m0_to_f32(s), 32, swizzled, None)
    else:
        want = O.mx_dequant(q, s, fmt, cols, swizzled=swizzled, cd=OUT[dtype])
    for off in (False, True):
        _check(K.dequantize_mx(_dev(q, off), _dev(s), elem, cols, swizzled=swizzled, dtype=dtype), want, dtype)


def test_swizzled_scale_offsets_beyond_32_bits() -> None:
    """One row of more than 2^29 columns: its swizzled scales are padded to 128 rows, 2^32 bytes and 512 more.  The last
    block's scales sit past 2^32, where an offset of 32 bits would read the first block's."""
    cols = (1 << 29) + 64
    q = torch.full((1, cols // 2), 0x22, dtype=torch.uint8, device="cuda")  # every code is 1.0
    s = torch.full((32, cols // 64 * 16), 0x38, dtype=torch.uint8, device="cuda")  # 1.0
    assert s.numel() == (1 << 32) + 512
    s.view(-1)[:4] = 0x30  # 0.5
    s.view(-1)[1 << 32:(1 << 32) + 4] = 0x40  # 2.0
    got = K.dequantize_nvfp4(q, s.view(torch.float8_e4m3fn), None, swizzled=True)[0]
    assert torch.equal(got[-64:].cpu(), torch.full((64,), 2.0, dtype=torch.bfloat16))
    assert torch.equal(got[:64].cpu(), torch.full((64,), 0.5, dtype=torch.bfloat16))
    assert bool((got[64:-64] == 1).all())
