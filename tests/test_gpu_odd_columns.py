"""Weights whose rows are no multiple of 16 elements (the general kernels' unaligned 16-byte accesses, and stochastic draws
whose Philox blocks straddle a lane's 16 elements) against the oracle, bit for bit: every offset of a row in its Philox
block, rows shorter than a lane's 16 elements, the last partial tile, both compute dtypes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import assert_merged_close, bf16_np, lora_factors, normal_bf16, oracle_dense_merge, u8_np
from piper_offload_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(9, 13), (17, 77), (33, 1003), (18, 4101), (5, 200)]


def _kw(dtype: torch.dtype, sr: bool) -> tuple[int | None, dict]:
    seed = 0xC0FFEE1234567 if sr else None
    return seed, {"cd": O.DT_F16 if dtype is torch.float16 else O.DT_BF16,
                  "sr_mode": O.SR_PHILOX8 if sr else O.SR_OFF, "seed": seed or 0}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("layout", ["row", "tensor"])
@pytest.mark.parametrize("shape", SHAPES)
def test_int8(shape: tuple[int, int], layout: str, sr: bool, dtype: torch.dtype) -> None:
    rows, cols = shape
    block = (1, cols) if layout == "row" else shape
    nq = rows if layout == "row" else 1
    rng = np.random.default_rng(rows * cols)
    q = torch.from_numpy(rng.integers(-128, 128, shape).astype(np.int8)).cuda()
    s = torch.from_numpy(rng.uniform(1e-4, 3e-4, (nq, 1)).astype(np.float32)).cuda()
    z = torch.from_numpy(rng.integers(-20, 20, (nq, 1)).astype(np.int8)).cuda()
    b, a = (t.cuda() for t in lora_factors(rows, cols, 16, 3, dtype=dtype))
    seed, kw = _kw(dtype, sr)
    for zp in (None, z):
        dense = K.dequantize_int8(q, s, zp, block, dtype=dtype, lora=(b, a, 0.75))
        oq, os_, oz = O.int8_requant(bf16_np(dense), cols if layout == "row" else rows * cols, asymmetric=zp is not None, **kw)
        gq, gs, gz = K.merge_int8_lora(q, s, zp, block, b, a, 0.75, asymmetric=zp is not None, reduce_range=False,
                                       rounding_seed=seed)
        assert np.array_equal(gq.cpu().numpy(), oq)
        assert np.array_equal(gs.cpu().numpy().reshape(-1), os_)
        assert np.array_equal(gz.cpu().numpy().reshape(-1), oz)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("layout", ["row", "tensor"])
@pytest.mark.parametrize("shape", SHAPES)
def test_fp8(shape: tuple[int, int], layout: str, sr: bool, dtype: torch.dtype) -> None:
    rows, cols = shape
    block = (1, cols) if layout == "row" else shape
    w = normal_bf16(shape, 0.02, rows).float()
    s = (w.abs().amax(1, keepdim=True) if layout == "row" else w.abs().amax().reshape(1, 1)) / 448
    q, s = (w / s).to(torch.float8_e4m3fn).cuda(), s.cuda()
    b, a = (t.cuda() for t in lora_factors(rows, cols, 16, 5, dtype=dtype))
    seed, kw = _kw(dtype, sr)
    dense = K.dequantize_float8(q, s, block, dtype=dtype, lora=(b, a, 0.75))
    oq, os_ = O.fp8_requant(bf16_np(dense), cols if layout == "row" else rows * cols, **kw)
    gq, gs = K.merge_float8_lora(q, s, block, b, a, 0.75, rounding_seed=seed)
    assert np.array_equal(u8_np(gq), oq)
    assert np.array_equal(gs.cpu().numpy().reshape(-1), os_)


@pytest.mark.parametrize("rank", [7, 64])
@pytest.mark.parametrize("shape", [*SHAPES, (70, 136)])
def test_dense(shape: tuple[int, int], rank: int) -> None:
    """Odd columns, an odd row stride, and whole pieces that end inside a column tile."""
    rows, cols = shape
    w = normal_bf16(shape, 0.02, cols)
    b, a = lora_factors(rows, cols, rank, 9)
    want = oracle_dense_merge(bf16_np(w), b, a, 0.75)
    for pad in (0, 3, 8):
        store = torch.zeros((rows, cols + pad), dtype=torch.bfloat16, device="cuda")
        store[:, :cols] = w.cuda()
        K.merge_dense_lora_(store[:, :cols], b.cuda(), a.cuda(), 0.75)
        assert_merged_close(bf16_np(store[:, :cols]), want, bf16_np(w))
        assert not store[:, cols:].any()  # nothing past the rows is written
