"""The no-allocation matmul where the reported workspace sits at its bound: accepted, and equal
bit for bit to the workspace entry point."""

from __future__ import annotations

import pytest
import torch

from test_zz_no_alloc import SCRATCH, _run_pair, announce

pytestmark = pytest.mark.gpu


# token chunks whose planes just fill the scratch; a K that is cut in parts
@pytest.mark.parametrize("M,N,K", [(16384, 300, 3072), (4096, 512, 28672)])
def test_float32_planes(gpu, M, N, K):
    announce(f"noalloc float32 planes M={M} N={N} K={K}")
    c_na, c_ws, need = _run_pair(gpu, M, N, K, torch.float32, seed=M + N)
    assert 0 < need <= SCRATCH
    assert torch.equal(c_na.view(torch.int32), c_ws.view(torch.int32))


# 384-row tiles, which use no workspace, and an image whose split would pass the scratch
@pytest.mark.parametrize("M,N,K,dtype", [(777, 9216, 3072, torch.bfloat16),
                                         (1024, 9216, 3072, torch.bfloat16),
                                         (512, 8448, 4096, torch.bfloat16),
                                         (65, 14336, 2048, torch.bfloat16),
                                         (1536, 6144, 4096, torch.int8),
                                         (1024, 9216, 3072, torch.int8)])
def test_tiles_and_images(gpu, M, N, K, dtype):
    announce(f"noalloc tiles and images M={M} N={N} K={K} {dtype}")
    c_na, c_ws, need = _run_pair(gpu, M, N, K, dtype, seed=M + N)
    assert need <= SCRATCH
    assert torch.equal(c_na.view(torch.int32), c_ws.view(torch.int32))
