"""K3's one round of 384 x 128 tiles (three row blocks per wave): bf16 and int8.

Exact against a float64 product of the unpacked trits on the GPU with integer activations
(every partial sum an integer below 2^24): last row tiles of 1 and 383 rows, a last token
tile of one token, one k-step, odd and even step counts, K past the last whole limb pair,
N that takes no 16-byte stores, C accumulated.
"""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import _lib, ops
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu

# M, N, K; 128..256 tiles of 384 x 128
CASES = [(700, 384 * 30 + 1, 208), (1000, 384 * 20 + 383, 96), (1025, 6000, 4112), (897, 9218, 3072),
         (129, 384 * 100, 304), (2048, 4096, 2000)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.int8])
@pytest.mark.parametrize("M,N,K", CASES)
def test_round_of_384_row_tiles(gpu, M, N, K, dtype):
    announce(f"384-row tiles M={M} N={N} K={K} {dtype}")
    assert 128 <= -(-N // 384) * -(-M // 128) <= 256
    g = torch.Generator("cpu").manual_seed(M + N + K)
    packed = ops.quantize_pack(torch.randn((N, K), generator=g).to(gpu), 0.45, _lib.THR_CPP)
    x = torch.randint(-127, 128, (M, K), generator=g).to(gpu)
    want = x.double() @ ops.unpack(packed, N, K).double().t().contiguous()
    c = torch.randint(-1000, 1001, (M, N), generator=g).to(gpu)
    xd = x.to(dtype)
    out = ops.ternary_matmul(xd, packed, K)
    assert torch.equal(out.double(), want)
    if dtype == torch.int8:
        out = ops.ternary_matmul(xd, packed, K, beta=1.0, c=c.to(torch.int32))
        assert torch.equal(out.double(), want + c.double())
    else:
        bias = torch.randint(-1000, 1001, (N,), generator=g).float().to(gpu)
        out = ops.ternary_matmul(xd, packed, K, alpha=0.5, beta=1.0, c=c.float(), bias=bias)
        assert torch.equal(out.double(), 0.5 * want + c.double() + bias.double())
