"""The training products where float32 overflows: as a float32 product gives them.

The products run as sums over bf16 planes, which must not overflow where the float32 sum does
not (a hi plane rounds up), and must come out as the infinity, never as infinity - infinity,
where it does.
"""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import qat
from test_gpu_exact_f32 import announce
from test_gpu_qat import PRODUCTS, U32

pytestmark = pytest.mark.gpu


def signed(gen, shape, lo, hi, gpu):
    v = lo + (hi - lo) * torch.rand(shape, generator=gen)
    return (v * (torch.randint(0, 2, shape, generator=gen) * 2 - 1)).to(gpu)


@pytest.mark.parametrize("M,N,K", PRODUCTS)
def test_weight_product_overflow(gpu, monkeypatch, M, N, K):
    """Finite operands.  One product of an output's sum past the largest float32 makes it that
    infinity (adding finite terms leaves it); a sum that passes it makes it too; a product just
    below it stays finite."""
    announce(f"qat weight product overflow M={M} N={N} K={K}")
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    gen = torch.Generator("cpu").manual_seed(M * 3 + N + K)
    g = torch.randn((M, N), generator=gen).to(gpu)
    x = torch.randn((M, K), generator=gen).to(gpu)
    m, ns, ks = M // 2, slice(N // 3, N), slice(K // 2, K)
    g[m, ns] = signed(gen, g[m, ns].shape, 1e25, 9e25, gpu)
    x[m, ks] = signed(gen, x[m, ks].shape, 1e25, 9e25, gpu)
    got, want = qat.weight_product(g, x), (g.double().T @ x.double())
    big = torch.zeros((N, K), dtype=torch.bool, device=gpu)
    big[ns, ks] = True
    assert torch.equal(got[big], torch.sign(want[big]).float() * float("inf"))
    mags = g.double().abs().T @ x.double().abs()
    assert bool(((got.double() - want).abs() <= 2.0 * (6 * M + 4) * U32 * mags + 1e-30)[~big].all())

    g, x = torch.full((M, N), 1e19, device=gpu), torch.full((M, K), -1e19, device=gpu)
    got = qat.weight_product(g, x)  # each product 1e38
    assert bool((got == -float("inf")).all()) if M > 3 else bool(got.isfinite().all())

    # hi planes round up: their product is 2^128, the value 2^128 (1 - 2^-8)
    g = torch.zeros((M, N), device=gpu)
    g[M - 1] = 2.0 ** 64 * (1 - 2.0 ** -9)
    x = torch.full((M, K), 2.0 ** 64 * (1 - 2.0 ** -9), device=gpu)
    want = 2.0 ** 128 * (1 - 2.0 ** -9) ** 2
    got = qat.weight_product(g, x).double()
    assert bool(((got - want).abs() <= 12 * U32 * want).all())
