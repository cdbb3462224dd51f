"""Encode of dense weights (csrc/lm_requant.h) against the oracle, bit for bit: rows that take 1 to 16 waves and one past
the register limit, few and many short rows, groups of every lane count and one that is no power of two, whole tensors with
odd sizes, block formats that end inside a workgroup, dense inputs that are not 16-byte aligned, more than one round per
workgroup, largest and smallest values, infinities and NaN."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import u8_np
from piper_offload_amd import kernels as K

pytestmark = pytest.mark.gpu

CD = {torch.bfloat16: O.DT_BF16, torch.float16: O.DT_F16}
FP4 = getattr(torch, "float4_e2m1fn_x2", None)


def _dense(shape: tuple[int, int], dtype: torch.dtype, offset: int = 0) -> tuple[torch.Tensor, np.ndarray]:
    g = torch.Generator().manual_seed(shape[0] * 7919 + shape[1])
    w = (torch.randn(shape, generator=g) * 0.02).to(dtype)
    w[0, : shape[1] // 2] = 0
    w[-1] *= 1000
    w[shape[0] // 2, 0] = -0.0
    flat = torch.empty(w.numel() + offset, dtype=dtype, device="cuda")
    flat[offset:] = w.reshape(-1).cuda()
    return flat[offset:].view(shape), w.view(torch.int16).numpy().view(np.uint16)


def _sr(sr: bool) -> tuple[int | None, dict]:
    seed = 0x9E3779B97F4A7C15
    return (seed, {"sr_mode": O.SR_PHILOX8, "seed": seed}) if sr else (None, {})


ROWS = [(5, 8), (300, 16), (4500, 16), (70, 64), (4097, 64), (4097, 72), (9, 512), (4, 1016), (3, 264), (9, 4096), (2, 4104), (2, 8200), (2, 16392), (2, 32776), (1, 65536), (2, 65544), (4, 77)]


def _blocks(shape: tuple[int, int]) -> list[tuple[tuple[int, int], int]]:
    rows, cols = shape
    out = [((1, cols), cols), ((rows, cols), rows * cols)]
    return out + [((1, g), g) for g in (16, 32, 64, 128, 192, 256, 512) if g < cols and cols % g == 0]


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("dtype", list(CD))
@pytest.mark.parametrize("shape", [*ROWS, (33, 1536), (6, 1024)])
def test_int8(shape: tuple[int, int], dtype: torch.dtype, sr: bool) -> None:
    seed, kw = _sr(sr)
    for offset in (0, 1):
        w, bits = _dense(shape, dtype, offset)
        for block, g in _blocks(shape):
            for asym, sdt in ((False, torch.float32), (True, torch.bfloat16)):
                q, s, z = K.requantize_int8(w, block, scale_dtype=sdt, asymmetric=asym, rounding_seed=seed)
                oq, os_, oz = O.int8_requant(bits, g, cd=CD[dtype], asymmetric=asym,
                                             scale_dt=O.DT_F32 if sdt is torch.float32 else O.DT_BF16, **kw)
                assert np.array_equal(q.cpu().numpy(), oq), (block, offset)
                s = s.cpu().reshape(-1)
                assert np.array_equal(s.numpy() if sdt is torch.float32 else s.view(torch.int16).numpy().view(np.uint16), os_)
                assert np.array_equal(z.cpu().numpy().reshape(-1), oz)


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("dtype", list(CD))
@pytest.mark.parametrize("shape", [*ROWS, (33, 1536), (6, 1024)])
def test_fp8(shape: tuple[int, int], dtype: torch.dtype, fp8: torch.dtype, sr: bool) -> None:
    seed, kw = _sr(sr)
    fmt = O.DT_E4M3 if fp8 is torch.float8_e4m3fn else O.DT_E5M2
    for offset in (0, 1):
        w, bits = _dense(shape, dtype, offset)
        for block, g in _blocks(shape):
            q, s = K.requantize_float8(w, block, fp8_dtype=fp8, rounding_seed=seed)
            oq, os_ = O.fp8_requant(bits, g, fmt=fmt, cd=CD[dtype], **kw)
            assert np.array_equal(u8_np(q), oq), (block, offset)
            assert np.array_equal(s.cpu().numpy().reshape(-1), os_)


BLOCKS = [(1, 32), (3, 96), (33, 160), (65, 2080)]


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("swizzled", [False, True])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", BLOCKS)
def test_block_formats(shape: tuple[int, int], offset: int, swizzled: bool, sr: bool) -> None:
    seed, kw = _sr(sr)
    w, bits = _dense(shape, torch.bfloat16, offset)
    for two in (False, True):
        q, s, p = K.requantize_nvfp4(w, two_level=two, swizzled=swizzled, rounding_seed=seed)
        oq, os_, op = O.nvfp4_requant(bits, two_level=two, swizzled=swizzled, **kw)
        assert np.array_equal(u8_np(q), oq)
        assert np.array_equal(u8_np(s), os_)
        assert not two or p.item() == op[0]
    for elem, fmt in ((FP4, O.DT_E2M1), (torch.float8_e4m3fn, O.DT_E4M3), (torch.float8_e5m2, O.DT_E5M2)):
        for mode in (0, 1, 2, 3):
            q, s = K.requantize_mx(w, elem, scaling_mode=mode, swizzled=swizzled, rounding_seed=seed)
            oq, os_ = O.mx_requant(bits, fmt, mode, swizzled=swizzled, **kw)
            assert np.array_equal(u8_np(q), oq)
            assert np.array_equal(u8_np(s), os_)
    if not swizzled:
        assert np.array_equal(u8_np(K.requantize_q8_0(w, rounding_seed=seed)), O.q8_0_requant(bits, **kw))


@pytest.mark.parametrize("sr", [False, True])
def test_several_rounds_per_workgroup(sr: bool) -> None:
    """More than 2^24 elements, so that the capped grids of the per-tensor maximum, the per-tensor encode and the two-level
    NVFP4 encode go round again: an odd count, and whole blocks."""
    seed, kw = _sr(sr)
    shape = (4097, 4099)
    n = shape[0] * shape[1]
    w, bits = _dense(shape, torch.bfloat16)
    q, s, _ = K.requantize_int8(w, shape, rounding_seed=seed)
    oq, os_, _ = O.int8_requant(bits, n, cd=O.DT_BF16, scale_dt=O.DT_F32, **kw)
    assert np.array_equal(q.cpu().numpy(), oq) and s.item() == os_[0]
    q, s = K.requantize_float8(w, shape, rounding_seed=seed)
    oq, os_ = O.fp8_requant(bits, n, fmt=O.DT_E4M3, cd=O.DT_BF16, **kw)
    assert np.array_equal(u8_np(q), oq) and s.item() == os_[0]
    w, bits = _dense((4100, 4112), torch.bfloat16)
    q, s, p = K.requantize_nvfp4(w, two_level=True, swizzled=False, rounding_seed=seed)
    oq, os_, op = O.nvfp4_requant(bits, two_level=True, swizzled=False, **kw)
    assert np.array_equal(u8_np(q), oq) and np.array_equal(u8_np(s), os_) and p.item() == op[0]


# A NaN is left out of maxima and encoded as the codes' lower limit (INT8: qmin).  An infinite value gives an infinite
# scale, whose codes only symmetric INT8, two-level NVFP4, MX and Q8_0 define (the others divide infinity by it).
@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("kind", ["largest", "smallest", "infinite", "nan"])
@pytest.mark.parametrize("dtype", list(CD))
@pytest.mark.parametrize("shape", [(40, 768), (5, 77), (3, 2048)])
def test_ends_of_the_range(shape: tuple[int, int], dtype: torch.dtype, kind: str, sr: bool) -> None:
    seed, kw = _sr(sr)
    rows, cols = shape
    info = torch.finfo(dtype)
    values = {"largest": [info.max, -info.max], "smallest": [info.tiny, -info.tiny / 2, 0.0, -0.0],
              "infinite": [float("inf"), -float("inf")], "nan": [float("nan")]}[kind]
    g = torch.Generator().manual_seed(cols)
    host = (torch.randn(shape, generator=g) * 0.02).to(dtype)
    at = torch.randint(0, host.numel(), (host.numel() // 40,), generator=g)
    host.view(-1)[at] = torch.tensor(values).to(dtype)[torch.randint(0, len(values), at.shape, generator=g)]
    w, bits = host.cuda(), host.view(torch.int16).numpy().view(np.uint16)
    finite = kind != "infinite"
    for block, group in [((1, cols), cols), (shape, rows * cols)] + ([((1, 64), 64)] if cols % 64 == 0 else []):
        for asym in (False, True) if finite else (False,):
            q, s, z = K.requantize_int8(w, block, asymmetric=asym, rounding_seed=seed)
            oq, os_, oz = O.int8_requant(bits, group, cd=CD[dtype], asymmetric=asym, scale_dt=O.DT_F32, **kw)
            assert np.array_equal(q.cpu().numpy(), oq), (block, asym)
            assert np.array_equal(s.cpu().numpy().reshape(-1), os_) and np.array_equal(z.cpu().numpy().reshape(-1), oz)
        for fp8, fmt in ((torch.float8_e4m3fn, O.DT_E4M3), (torch.float8_e5m2, O.DT_E5M2)) if finite else ():
            q, s = K.requantize_float8(w, block, fp8_dtype=fp8, rounding_seed=seed)
            oq, os_ = O.fp8_requant(bits, group, fmt=fmt, cd=CD[dtype], **kw)
            assert np.array_equal(u8_np(q), oq), (block, fp8)
            assert np.array_equal(s.cpu().numpy().reshape(-1), os_)
    if cols % 32 or dtype is not torch.bfloat16:
        return
    for two in (False, True) if finite else (True,):
        q, s, p = K.requantize_nvfp4(w, two_level=two, swizzled=False, rounding_seed=seed)
        oq, os_, op = O.nvfp4_requant(bits, two_level=two, swizzled=False, **kw)
        assert np.array_equal(u8_np(q), oq) and np.array_equal(u8_np(s), os_), two
        assert not two or p.item() == op[0]
    for elem, fmt in ((FP4, O.DT_E2M1), (torch.float8_e4m3fn, O.DT_E4M3), (torch.float8_e5m2, O.DT_E5M2)):
        for mode in (0, 1, 2, 3):
            q, s = K.requantize_mx(w, elem, scaling_mode=mode, swizzled=False, rounding_seed=seed)
            oq, os_ = O.mx_requant(bits, fmt, mode, swizzled=False, **kw)
            assert np.array_equal(u8_np(q), oq) and np.array_equal(u8_np(s), os_), (elem, mode)
    assert np.array_equal(u8_np(K.requantize_q8_0(w, rounding_seed=seed)), O.q8_0_requant(bits, **kw))
