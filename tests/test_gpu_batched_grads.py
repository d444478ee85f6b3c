"""Batched gradients (several output gradients through one graph at once, as vectorized Jacobians
take them) of layers whose backward runs on kernels elsewhere."""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import nn as t8nn, qat
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu


def batched(y, inputs, v):
    return torch.autograd.grad(y, inputs, v, is_grads_batched=True, retain_graph=True)


def vmapped(y, inputs, v):
    return torch.func.vmap(lambda g: torch.autograd.grad(y, inputs, g, retain_graph=True))(v)


@pytest.mark.parametrize("take", [batched, vmapped])
@pytest.mark.parametrize("kernels", [False, True])
def test_training_layer(gpu, monkeypatch, take, kernels):
    announce(f"batched gradients, training, {take.__name__} {kernels}")
    if kernels:
        monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
        monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    torch.manual_seed(2)
    layer = t8nn.Linear(48, 40, device=gpu).train()
    x = torch.randn((80, 48), device=gpu, requires_grad=True)
    y = layer(x)
    inputs = [x, layer.weight, layer.bias]
    v = torch.randn((3, *y.shape), device=gpu)
    got = take(y, inputs, v)
    for i in range(3):
        for a, b in zip(got, torch.autograd.grad(y, inputs, v[i], retain_graph=True)):
            torch.testing.assert_close(a[i], b, rtol=1e-5, atol=1e-5)
    jac = torch.autograd.functional.jacobian(lambda z: layer(z).sum(0), x.detach(), vectorize=True)
    assert jac.shape == (40, 80, 48) and bool(jac.isfinite().all())


@pytest.mark.parametrize("take", [batched, vmapped])
def test_frozen_layers_bias(gpu, take):
    announce(f"batched gradients, frozen bias, {take.__name__}")
    layer = t8nn.Linear(48, 40, device=gpu).eval()
    y = layer(torch.randn((7, 48), device=gpu))
    v = torch.randn((3, *y.shape), device=gpu)
    (got,) = take(y, [layer.bias], v)
    torch.testing.assert_close(got, v.sum(1), rtol=1e-5, atol=1e-5)
