"""A training forward reads its weight twice: once for the scale, once for its trits.  A weight
that a parametrization computes may draw random numbers or move its own state at each read."""

from __future__ import annotations

import pytest
import torch
from torch import nn
from torch.nn.utils import parametrize

from t81lib_amd import nn as t8nn

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


class Counted(nn.Module):
    calls = 0

    def forward(self, w):
        self.calls += 1
        return w * 1.0


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("stochastic", [False, True])
def test_reads_per_forward(device, stochastic):
    layer = t8nn.Linear(48, 40, device=device).train()
    layer.configure_qat(stochastic_rounding=stochastic)
    count = Counted()
    parametrize.register_parametrization(layer, "weight", count)
    count.calls = 0
    layer(torch.randn((5, 48), device=device)).sum().backward()
    assert count.calls == 2
    assert layer.parametrizations.weight.original.grad is not None


@pytest.mark.parametrize("device", DEVICES)
def test_random_weight_repeats(device):
    """The draws of a weight that is random at each read, in the expression's order."""

    class Dropped(nn.Module):
        def forward(self, w):
            return nn.functional.dropout(w, 0.5)

    layer = t8nn.Linear(48, 40, device=device).train()
    parametrize.register_parametrization(layer, "weight", Dropped())
    x = torch.randn((5, 48), device=device)
    torch.manual_seed(3)
    got = layer(x)
    torch.manual_seed(3)
    scale = layer.weight.detach().abs().amax().clamp(min=1e-6)
    u = layer.weight / scale
    q = torch.where(u.abs() >= layer.ternary_threshold, u.sign(), torch.zeros_like(u))
    want = nn.functional.linear(x, q * scale, layer.bias)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("device", DEVICES)
def test_replaced_on_one_layer(device):
    """A layer whose own quantizer a program replaced uses it."""
    layer = t8nn.Linear(48, 40, bias=False, device=device).train()
    layer._quantize_training_weight = lambda: torch.ones((40, 48), device=device)
    x = torch.randn((5, 48), device=device)
    assert torch.equal(layer(x), nn.functional.linear(x, torch.ones((40, 48), device=device)))
