"""Q8_0 merges of csrc/lm_q8_fast.h, whose waves keep one column tile and walk down its row groups, against the oracle's
requant of the GPU's dense merge, byte for byte and in place: a weight with several row groups per wave and a ragged last
one, a single tile, and rows so long that the tiles alone fill the GPU (8 waves per tile, more than are resident)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import bf16_np, lora_factors, normal_bf16, u8_np
from piper_offload_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank", [16, 32, 64])
@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("shape", [(4105, 1920), (1, 128), (70003, 128), (200, 66560)])
def test_merge_equals_oracle(shape: tuple[int, int], sr: bool, rank: int) -> None:
    rows, cols = shape
    packed = torch.from_numpy(O.q8_0_requant(bf16_np(normal_bf16(shape, 0.02, rows)))).cuda()
    b, a = (t.cuda() for t in lora_factors(rows, cols, rank, rank))
    seed = 0x1234567890ABCDEF if sr else None
    dense = K.dequantize_gguf(packed, 8, lora=(b, a, 0.75))
    ref = O.q8_0_requant(bf16_np(dense), sr_mode=O.SR_PHILOX8 if sr else O.SR_OFF, seed=seed or 0)
    K.merge_q8_0_lora(packed, b, a, 0.75, rounding_seed=seed, out=packed)
    assert np.array_equal(u8_np(packed), ref)
