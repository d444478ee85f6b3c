"""The plane-image product of K3 (gemm_planes.hip): float32 activations as bf16 planes.

Bit-exact against the integer oracle with fixed-point activations (both planes exact, every
partial sum exact in float32), at the sizes where tiles, pieces, splits and epilogues end:
one limb pair, an odd limb count, K that is no multiple of 8 (the last 16-byte piece is
part zeros), a last token block of one token, row tiles of one row, N that is no multiple of
4 (scalar epilogue), K split over the workspace, x off 16-byte alignment.
"""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import _lib, ops
from test_gpu_exact_f32 import announce, run_cases

pytestmark = pytest.mark.gpu

# M, K, N, elements x is off 16-byte alignment
EDGES = [(65, 8, 513, 0), (33, 97, 512, 0), (64, 1001, 511, 1), (129, 144, 5, 0), (97, 4001, 1030, 0),
         (34, 4100, 1025, 0), (160, 2000, 1536, 3), (257, 96, 2052, 0), (65, 9000, 130, 0)]


@pytest.mark.parametrize("M,K,N,offset", EDGES)
def test_planes_bit_exact(gpu, orc, M, K, N, offset):
    announce(f"planes M={M} K={K} N={N} offset={offset}")
    assert _lib.lib().t81_hip_ternary_matmul_workspace_size(M, N, K, _lib.DTYPE_F32) > 0
    run_cases(gpu, orc, M, N, K, seed=M * 31 + K + N, kernel=3, what="planes", offset=offset)


def test_planes_keep_tokens_apart(gpu):
    """An infinity or NaN in one token reaches that token's outputs only (pieces and tokens
    that do not exist are zeros, not a neighbour's values)."""
    M, K, N = 70, 1001, 600
    announce("planes non-finite tokens")
    g = torch.Generator("cpu").manual_seed(3)
    packed = ops.quantize_pack(torch.randn((N, K), generator=g).to(gpu), 0.45, _lib.THR_CPP)
    x = torch.randn((M, K), generator=g).to(gpu)
    clean = ops.ternary_matmul(x, packed, K)
    x[3, K - 1] = float("inf")
    x[69, 0] = float("nan")
    y = ops.ternary_matmul(x, packed, K)
    rest = [m for m in range(M) if m not in (3, 69)]
    assert torch.equal(y[rest], clean[rest])
    assert torch.isnan(y[69]).all() and not torch.isfinite(y[3]).any()
