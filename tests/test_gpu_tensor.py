"""Per-tensor FP8 and INT8 merges through csrc/lm_tensor.hip against the oracle's requant of the GPU's dense merge, bit for
bit and in place: ragged rows, column counts that leave waves without tiles, every rank bucket and all wave tilings of
each, a weight too short for its row length (which the general kernels take), odd columns and fp16 factors (likewise)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import bf16_np, fp8_initial, lora_factors, normal_bf16, u8_np
from piper_offload_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(2, 64), (17, 128), (65, 4160), (130, 8256), (300, 2112), (2, 65600), (40, 200)]


@pytest.mark.parametrize("rank", [5, 32, 64])
@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2", "int8"])
@pytest.mark.parametrize("shape", SHAPES)
def test_merge_equals_oracle(shape: tuple[int, int], fmt: str, sr: bool, rank: int) -> None:
    _case(shape, fmt, sr, rank, torch.bfloat16)


def test_rank_64_large() -> None:
    _case((8208, 8192), "e4m3", True, 64, torch.bfloat16)


@pytest.mark.parametrize("fmt", ["e4m3", "int8"])
def test_fp16_factors(fmt: str) -> None:
    _case((70, 256), fmt, False, 16, torch.float16)


def _case(shape: tuple[int, int], fmt: str, sr: bool, rank: int, dtype: torch.dtype) -> None:
    rows, cols = shape
    w = normal_bf16(shape, 0.02, rows + cols)
    b, a = (t.cuda() for t in lora_factors(rows, cols, rank, rank, dtype=dtype))
    seed = 0x1234567890ABCDEF if sr else None
    kw = {"cd": O.DT_F16 if dtype is torch.float16 else O.DT_BF16,
          "sr_mode": O.SR_PHILOX8 if sr else O.SR_OFF, "seed": seed or 0}
    if fmt == "int8":
        s = (w.float().abs().amax() / 127).reshape(1, 1)
        q, s = torch.round(w.float() / s).clamp(-128, 127).to(torch.int8).cuda(), s.cuda()
        dense = K.dequantize_int8(q, s, None, shape, dtype=dtype, lora=(b, a, 0.75))
        oq, os_, _ = O.int8_requant(bf16_np(dense), rows * cols, **kw)
        z = torch.full((1, 1), 3, dtype=torch.int8, device="cuda")
        K.merge_int8_lora_into(q, s, None, shape, b, a, 0.75, asymmetric=False, reduce_range=False, rounding_seed=seed,
                               out_qdata=q, out_scale=s, out_zero_point=z)
        assert z.item() == 0
    else:
        fp8 = torch.float8_e4m3fn if fmt == "e4m3" else torch.float8_e5m2
        flat, s = fp8_initial(w.reshape(1, -1), fp8)
        q, s = flat.reshape(shape).cuda(), s.cuda()
        dense = K.dequantize_float8(q, s, shape, dtype=dtype, lora=(b, a, 0.75))
        oq, os_ = O.fp8_requant(bf16_np(dense), rows * cols, fmt=O.DT_E4M3 if fmt == "e4m3" else O.DT_E5M2, **kw)
        K.merge_float8_lora_into(q, s, shape, b, a, 0.75, rounding_seed=seed, out_qdata=q, out_scale=s)
    assert np.array_equal(u8_np(q), oq.view(np.uint8))
    assert s.item() == os_[0]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape", [(70, 256), (40, 200)])
def test_symmetric_with_zero_point(shape: tuple[int, int], in_place: bool) -> None:
    """A zero point that comes with a symmetric request is subtracted, as in the dense merge; the merged codes have none."""
    rows, cols = shape
    rank = 8
    g = torch.Generator().manual_seed(7)
    q = torch.randint(-100, 100, (rows, cols), generator=g, dtype=torch.int8).cuda()
    s, z = torch.full((1, 1), 3e-4, device="cuda"), torch.full((1, 1), 5, dtype=torch.int8, device="cuda")
    b, a = (t.cuda() for t in lora_factors(rows, cols, rank, rank))
    dense = K.dequantize_int8(q, s, z, (rows, cols), lora=(b, a, 0.75))
    oq, os_, _ = O.int8_requant(bf16_np(dense), rows * cols)
    out_q, out_s, out_z = (q, s, z) if in_place else (torch.empty_like(q), torch.empty_like(s), torch.empty_like(z))
    K.merge_int8_lora_into(q, s, z, (rows, cols), b, a, 0.75, asymmetric=False, reduce_range=False, rounding_seed=None,
                           out_qdata=out_q, out_scale=out_s, out_zero_point=out_z)
    assert np.array_equal(u8_np(out_q), oq.view(np.uint8))
    assert out_s.item() == os_[0] and out_z.item() == 0


@pytest.mark.parametrize("rank", [5, 32, 64])
@pytest.mark.parametrize("fmt,sr", [("e4m3", True), ("int8", False)])
@pytest.mark.parametrize("shape", [(130, 65600), (4100, 2112), (2047, 4096), (2048, 4096)])
def test_from_2_to_the_23rd_elements(shape: tuple[int, int], fmt: str, sr: bool, rank: int) -> None:
    """The larger wave tiles: ragged rows and column counts, and either side of the line between them and the small ones."""
    _case(shape, fmt, sr, rank, torch.bfloat16)
