"""The single-factor up projection in whole cache lines and the down projection's column pairs (csrc/lm_routed.hip): last
token tiles of 1 to 15 rows, outputs narrower than a tile and of ragged width, input widths that end inside a pair or a
round, every chunk count.  Same oracle and bounds as test_gpu_routed.py; the output may alias y."""

from __future__ import annotations

import pytest
import torch

import test_gpu_routed
from piper_offload_amd.routed import RoutedFactor, routed_residual
from test_gpu_routed import _case, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,K,N,rank", [(17, 4160, 136, 32), (31, 100, 8, 16), (33, 4104, 72, 64), (129, 8232, 264, 24),
                                        (24, 36, 64, 4), (47, 1024, 200, 48), (300, 520, 1032, 16)])
def test_lean_up_matches_oracle(T: int, K: int, N: int, rank: int, dtype: torch.dtype, monkeypatch) -> None:
    # Elements that may differ at all: a value p = x A^T rounds the other way when its fp32 sum, taken in another order
    # (about 2^-22 relative apart), lies that close to a rounding boundary: with an ulp of 2^-10 (fp16) or 2^-7 (bf16), one
    # value in 2^11 or 2^14 or so, and it can move every output of its token.  Four times the expected share of tokens,
    # plus two tokens (these results have few).
    share = 4 * rank * 2.0 ** (-11 if dtype is torch.float16 else -14) + 2 / T
    monkeypatch.setattr(test_gpu_routed, "ROUTED_MISMATCH", max(test_gpu_routed.ROUTED_MISMATCH, share))
    x, y, fs = _case(T, K, N, [rank], False, dtype, T + K)
    dfs = [RoutedFactor(f.a.cuda(), f.b.cuda(), f.strength) for f in fs]
    with torch.no_grad():
        got = routed_residual(x.cuda(), dfs, y.cuda())
    _check(got, x, y, fs, dtype)
