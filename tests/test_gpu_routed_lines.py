"""The routed residual's tilings (csrc/lm_routed.hip), bit for bit against the oracle on inputs whose sums are exact: the
single-factor up projection in whole cache lines and the down projection's column pairs (last token tiles of 1 to 15 rows,
outputs narrower than a tile and of ragged width, input widths that end inside a pair or a round, every chunk count), the
down projection's shares, several token tiles per wave, and an output that aliases y.  test_gpu_routed.py has general
inputs."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from piper_offload_amd import _lib as L
from piper_offload_amd.routed import RoutedFactor, routed_residual
from test_gpu_routed import DT, _bits

pytestmark = pytest.mark.gpu


def _integer_case(T: int, K: int, N: int, ranks: list[int], bias: bool, dtype: torch.dtype, seed: int):
    """Inputs whose fp32 sums are exact in every order: x, A and b are small integers, so p = x A^T is an integer and p s a
    multiple of 1/4, both far below 2^16 (|p| < 6 sigma = 6 sqrt(4 K / 3)), and a sum of 64 products p s b spans under 24
    bits.  Only the roundings to the dtype are left, and those have one order: results equal the oracle bit for bit."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randint(-2, 3, (T, K), generator=g).to(dtype)
    y = (torch.randn(T, N, generator=g) * 64).to(dtype)
    fs = [RoutedFactor(torch.randint(-1, 2, (r, K), generator=g).to(dtype),
                       torch.randint(-2, 3, (N, r), generator=g).to(dtype), [1.0, 0.5, -1.25][i % 3],
                       torch.randn(N, generator=g).to(dtype) if bias else None) for i, r in enumerate(ranks)]
    return x, y, fs


def _oracle(x, y, fs, dtype) -> torch.Tensor:
    ref = O.routed_residual(_bits(x), _bits(y), [(_bits(f.a), _bits(f.b), None if f.bias is None else _bits(f.bias),
                                                  f.strength) for f in fs], dt=DT[dtype])
    return torch.from_numpy(ref.view(np.int16)).view(dtype)


def _cuda(fs):
    return [RoutedFactor(f.a.cuda(), f.b.cuda(), f.strength, None if f.bias is None else f.bias.cuda()) for f in fs]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,K,N,rank", [(17, 4160, 136, 32), (31, 100, 8, 16), (33, 4104, 72, 64), (129, 8232, 264, 24),
                                        (24, 36, 64, 4), (47, 1024, 200, 48), (300, 520, 1032, 16)])
def test_lean_up_matches_oracle(T: int, K: int, N: int, rank: int, dtype: torch.dtype) -> None:
    x, y, fs = _integer_case(T, K, N, [rank], False, dtype, T + K)
    with torch.no_grad():
        got = routed_residual(x.cuda(), _cuda(fs), y.cuda())
    assert torch.equal(got.cpu(), _oracle(x, y, fs, dtype))


# The down projection's shares (down_plan): K spans that end inside a step, chunk blocks of 1, 2 and 4 with a last one of
# fewer chunks, one span and many, more tiles than workgroups wanted; spans summed by a launch of their own and by both up
# kernels, for one token tile per wave and for two.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,K,N,ranks,bias", [(17, 14336, 72, [64, 64, 64, 64], False), (33, 4100, 200, [16], False),
                                              (130, 3080, 64, [8, 40, 64], True), (300, 9000, 136, [16], False),
                                              (1030, 2056, 72, [64], False), (1024, 7000, 64, [64], False),
                                              (1100, 6200, 40, [48, 16, 5], True), (2050, 1024, 64, [16, 16], False),
                                              (4100, 256, 64, [64], False), (17, 1024, 64, [1], False),
                                              (70, 9000, 1000, [16, 8], True), (40, 5000, 100, [16, 16, 9], False),
                                              (20, 12000, 136, [30], False), (637, 2100, 14336, [16], False),
                                              (637, 2100, 14336, [8], True)])
def test_down_projection_shares(T: int, K: int, N: int, ranks: list[int], bias: bool, dtype: torch.dtype) -> None:
    x, y, fs = _integer_case(T, K, N, ranks, bias, dtype, T + K)
    with torch.no_grad():
        got = routed_residual(x.cuda(), _cuda(fs), y.cuda())
    assert torch.equal(got.cpu(), _oracle(x, y, fs, dtype))


def _through_c_entry(x, fs, y, out) -> None:
    """lm_routed_residual on GPU tensors, with an output of the caller's (routed_residual allocates its own)."""
    arr = (L.RoutedFactor * len(fs))()
    for i, f in enumerate(fs):
        arr[i].a, arr[i].b, arr[i].bias = f.a.data_ptr(), f.b.data_ptr(), None if f.bias is None else f.bias.data_ptr()
        arr[i].strength, arr[i].rank = f.strength, f.a.shape[0]
    (t, k), n, h = x.shape, y.shape[1], L.lib()
    nbytes = h.lm_routed_workspace_size(t, k, arr, len(fs))
    ws = L.workspace(nbytes, x.device)
    L.check(h.lm_routed_residual(x.data_ptr(), y.data_ptr(), out.data_ptr(), t, k, n, L.torch_dtype_id(x.dtype), arr,
                                 len(fs), L.aligned_ptr(ws), nbytes, L.stream_ptr(x.device)))
    torch.cuda.synchronize()


# Up kernels that walk several token tiles per wave, the last one ragged, and single launches, into another tensor and in
# place: the output may alias y.  [1033, 14336]: 2 tiles per wave (one factor, and two with a bias), 4 at rank 64 and 80;
# N % 8 != 0 takes the element-wise stores.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,K,N,ranks,bias", [(1033, 72, 14336, [16], False), (1033, 72, 14336, [8, 24], True),
                                              (1033, 72, 14336, [64], False), (1033, 72, 14336, [64, 16], False),
                                              (2100, 40, 8196, [16], False), (47, 96, 200, [48], False),
                                              (9, 96, 136, [16], False), (16, 96, 100, [16, 24], True)])
def test_several_token_tiles_and_aliased_output(T: int, K: int, N: int, ranks: list[int], bias: bool,
                                                dtype: torch.dtype) -> None:
    x, y, fs = _integer_case(T, K, N, ranks, bias, dtype, T + N)
    ref, dx, dy, dfs = _oracle(x, y, fs, dtype), x.cuda(), y.cuda(), _cuda(fs)
    out = torch.empty_like(dy)
    _through_c_entry(dx, dfs, dy, out)
    assert torch.equal(out.cpu(), ref)
    assert torch.equal(dy.cpu(), y)
    _through_c_entry(dx, dfs, dy, dy)
    assert torch.equal(dy.cpu(), ref)
