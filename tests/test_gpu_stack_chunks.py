"""Grouped NVFP4 merges whose rows span several column chunks (csrc/lm_nvfp4_fast.h, nv_chunks): every target of a stack
equals its single-target merge, which test_gpu_nvfp4.py checks against the oracle.  Rows of one tile past a chunk, of the
tile counts that split unevenly, ragged row groups, one and two scale levels."""

from __future__ import annotations

import pytest
import torch

from helpers import lora_factors, normal_bf16
from piper_offload_amd import NVFP4Weight
from piper_offload_amd import kernels as K
from piper_offload_amd.stack import StackTarget, merge_nvfp4_stack

pytestmark = pytest.mark.gpu

SHAPES = [(33, 4224), (64, 128), (17, 14336), (96, 8320), (40, 4096), (1, 12416)]


@pytest.mark.parametrize("rank", [16, 32])
@pytest.mark.parametrize("swizzled", [False, True])
@pytest.mark.parametrize("sr", [False, True])
def test_chunked_rows_equal_single_merges(sr: bool, swizzled: bool, rank: int) -> None:
    _case(SHAPES, sr, swizzled, rank)


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("rows", [32 * 8187, 32 * 8186])
def test_swizzled_stacks_of_many_rows(rows: int, sr: bool) -> None:
    """8192 units of 32 rows keep whole rows (NV_WHOLE_ROWS), one unit less is chunked; the second target has rows of 33
    tiles, one past a chunk."""
    _case([(rows, 128), (33, 4224), (65, 128)], sr, True, 16)


def _case(shapes: list[tuple[int, int]], sr: bool, swizzled: bool, rank: int) -> None:
    targets, want = [], []
    for i, (rows, cols) in enumerate(shapes):
        w = normal_bf16((rows, cols), 0.02, i).cuda()
        q, s, p = K.requantize_nvfp4(w, two_level=i % 3 != 2, swizzled=swizzled)
        b, a = (t.cuda() for t in lora_factors(rows, cols, rank, 100 + i))
        want.append(K.merge_nvfp4_lora(q, s, p, 16, swizzled, b, a, 0.75, rounding_seed=77 + i if sr else None))
        targets.append(StackTarget(NVFP4Weight(q, s, p, 16, is_swizzled_scales=swizzled), b, a, 0.75, 77 + i))
    merge_nvfp4_stack(targets, stochastic=sr)
    for i, (t, (q, s, p)) in enumerate(zip(targets, want)):
        assert torch.equal(t.weight.qdata, q), shapes[i]
        assert torch.equal(t.weight.scale.view(torch.uint8), s.view(torch.uint8)), shapes[i]
        assert p is None or torch.equal(t.weight.per_tensor_scale, p)
