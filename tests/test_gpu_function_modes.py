"""A program's torch-function modes see the operations of a layer under autograd, as they do
where no kernel stands in; device contexts, which are such modes, do not turn the kernels off."""

from __future__ import annotations

import pytest
import torch
from torch.overrides import TorchFunctionMode

from t81lib_amd import nn as t8nn, qat
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu


class Seen(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(getattr(func, "__name__", str(func)))
        return func(*args, **(kwargs or {}))


def test_training_layer_under_function_modes(gpu, monkeypatch):
    announce("function modes, training")
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    layer = t8nn.Linear(48, 40, device=gpu).train()
    x = torch.randn((80, 48), device=gpu)
    with Seen() as seen:
        layer(x).sum().backward()
    assert "linear" in seen.names and "amax" in seen.names
    with torch.device(gpu):
        assert qat.product_on_kernels(x, layer.weight, layer.bias)
        with Seen() as seen:
            layer(x)
        assert "linear" in seen.names


def test_frozen_layer_under_function_modes(gpu):
    announce("function modes, frozen")
    layer = t8nn.Linear(48, 40, device=gpu).eval()
    x = torch.randn((7, 48), device=gpu, requires_grad=True)
    want = layer(x)
    with Seen() as seen:
        got = layer(x)
    assert torch.equal(got, want) and any("add" in n for n in seen.names)
