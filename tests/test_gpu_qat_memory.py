"""A training step on a device whose memory is nearly used up: where the kernels' workspaces do
not fit, the library's products, which need none, run as they did."""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import qat
from test_gpu_exact_f32 import announce
from test_gpu_matmul_memory import no_room_for
from test_gpu_qat import layers

pytestmark = pytest.mark.gpu


def test_step_without_room_for_workspaces(gpu, monkeypatch):
    announce("qat step near the memory limit")
    torch.manual_seed(4)
    layer = layers(4096, 4096, True, gpu)
    x = torch.randn((2048, 4096), device=gpu, requires_grad=True)
    g = torch.randn((2048, 4096), device=gpu)
    assert qat.product_on_kernels(x, layer.weight, layer.bias)

    def step():
        layer.training_scale = x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(g)
        return y.detach(), x.grad, layer.weight.grad, layer.bias.grad

    want = step()
    real, asked = qat._scratch, []

    def scratch(nbytes, device):
        with no_room_for(16 << 20, device):
            asked.append((nbytes, real(nbytes, device)))
        return asked[-1][1]

    monkeypatch.setattr(qat, "_scratch", scratch)
    got = step()
    assert len(asked) == 3 and all(n > 16 << 20 and ws is None for n, ws in asked)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.abs().max()))
