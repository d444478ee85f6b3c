"""The training products bit for bit, with each plane and each pair of planes needed at each tile
edge, tail and split (tests/test_plane_inputs.py shows on the CPU that they are)."""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import ops, qat
from test_gpu_exact_f32 import announce
from test_gpu_qat import PRODUCTS, STEPS
from test_plane_inputs import ternary_inputs, weight_product_inputs

pytestmark = pytest.mark.gpu


# (and several tiles of 256 x 256 with the rows split, more than a round of them)
@pytest.mark.parametrize("M,N,K", PRODUCTS + [(600, 1300, 1544), (40, 4100, 4360)])
def test_weight_product(gpu, monkeypatch, M, N, K):
    announce(f"plane pairs, weight product M={M} N={N} K={K}")
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    for kind, (g, x) in enumerate(weight_product_inputs(M, N, K)):
        got = qat.weight_product(g.to(gpu), x.to(gpu))
        want = g.to(gpu).double().T @ x.to(gpu).double()
        assert torch.equal(got.double(), want), f"kind {kind}: {int((got.double() != want).sum())}"


# (and several row and token tiles, more than a round of them, K in several steps)
@pytest.mark.parametrize("M,K,N", STEPS + [(300, 2000, 1537), (2050, 500, 16900)])
def test_ternary_product(gpu, M, K, N):
    """scale * (X T^T) + bias for scales whose products stay exact."""
    announce(f"planes, ternary product M={M} K={K} N={N}")
    x, t = (v.to(gpu) for v in ternary_inputs(M, K, N))
    packed = ops.quantize_pack(t, 0.5)
    want = x.double() @ t.double().T
    for s in (1.0, 0.0625, 4.0):
        scale = torch.tensor(s, device=gpu)
        got = qat._matmul(x, packed, N, scale, None)
        assert torch.equal(got.double(), s * want), f"scale {s}"
    bias = torch.randint(-9, 10, (N,), device=gpu).float()
    got = qat._matmul(x, packed, N, torch.tensor(1.0, device=gpu), bias)
    assert torch.equal(got.double(), want + bias.double())
