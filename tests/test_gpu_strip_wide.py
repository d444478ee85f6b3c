"""One token over wide outputs: the strip kernel's longer strips (14 and 16 loads).

Exact against a float64 product of the unpacked trits with integer activations (every partial
sum an integer below 2^24): the first and last widths of each strip length, a last strip of
one row and of one row short, K off the vector loads, C accumulated and a bias.
"""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import _lib, ops
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [3073, 4096, 4500, 4608])
@pytest.mark.parametrize("N", [16384, 16385, 28671, 28672, 28673, 32767, 32768, 32769])
def test_wide_strips(gpu, N, K):
    announce(f"wide strip N={N} K={K}")
    g = torch.Generator("cpu").manual_seed(N + K)
    packed = ops.quantize_pack(torch.randn((N, K), generator=g).to(gpu), 0.45, _lib.THR_CPP)
    x = torch.randint(-7, 8, (1, K), generator=g).to(gpu, torch.bfloat16)
    want = x.double() @ ops.unpack(packed, N, K).double().t().contiguous()
    out = ops.ternary_matmul(x, packed, K)
    assert torch.equal(out.double(), want)
    bias = torch.randint(-99, 100, (N,), generator=g).float().to(gpu)
    c = torch.randint(-99, 100, (1, N), generator=g).float().to(gpu)
    out = ops.ternary_matmul(x, packed, K, beta=1.0, c=c.clone(), bias=bias)
    assert torch.equal(out.double(), want + c.double() + bias.double())
