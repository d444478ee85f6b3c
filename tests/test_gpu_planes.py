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


# bf16 activations through their image: K that is no multiple of 8 (and x off alignment), few
# tokens over a split that does not fit, tokens and rows past a tile, one limb pair
BF16 = [(17, 8193, 4100, 0), (33, 1025, 1030, 0), (96, 97, 513, 1), (130, 1001, 512, 0),
        (100, 4096, 1030, 0), (129, 2048, 2052, 0), (200, 4096, 1536, 3), (65, 4104, 600, 0)]


@pytest.mark.parametrize("M,K,N,offset", BF16)
def test_bf16_image_bit_exact(gpu, orc, M, K, N, offset):
    """Integer activations |x| <= 127: every partial sum is an integer below 2^24."""
    announce(f"bf16 image M={M} K={K} N={N} offset={offset}")
    g = torch.Generator("cpu").manual_seed(M + K + N)
    packed = ops.quantize_pack(torch.randn((N, K), generator=g).to(gpu), 0.45, _lib.THR_CPP)
    xi = torch.randint(-127, 128, (M, K), generator=g)
    store = torch.zeros(M * K + 8, dtype=torch.bfloat16, device=gpu)
    x = store[offset:offset + M * K].view(M, K)
    x.copy_(xi.to(gpu))
    acc = torch.from_numpy(orc.trit_matmul_i64(xi.to(torch.int8).numpy(), packed.cpu().numpy(), K))
    c = torch.randint(-1000, 1001, (M, N), generator=g).float()
    bias = torch.randint(-1000, 1001, (N,), generator=g).float()
    for alpha, beta, use_bias in ((1.0, 0.0, False), (0.5, 1.0, True)):
        out = ops.ternary_matmul(x, packed, K, alpha=alpha, beta=beta,
                                 c=c.to(gpu) if beta else None,
                                 bias=bias.to(gpu) if use_bias else None)
        want = alpha * acc.double() + (beta * c.double() if beta else 0.0)
        if use_bias:
            want = want + bias.double()
        assert torch.equal(out.cpu().double(), want), f"alpha={alpha}"
