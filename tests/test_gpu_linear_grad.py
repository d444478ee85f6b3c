"""A frozen ternary layer under autograd: the fused bias, its gradient as column sums."""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import nn as t8nn, ops, tensor
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu

# rows around a run (64), several runs, more than 64 runs; columns around a block (64, 256)
SUMS = [(0, 5), (1, 1), (3, 64), (15, 257), (63, 256), (64, 65), (65, 4), (130, 1000), (1024, 258),
        (4096, 260), (4097, 63), (70000, 8)]


@pytest.mark.parametrize("rows,cols", SUMS)
def test_column_sum(gpu, rows, cols):
    """Any order of `rows` float32 additions is within rows 2^-24 sum |g| of the exact sum."""
    announce(f"column sum {rows}x{cols}")
    g = torch.randn((rows, cols), generator=torch.Generator("cpu").manual_seed(rows + cols)).to(gpu)
    for view in (g, torch.cat([g.new_zeros(1), g.reshape(-1)])[1:].view(rows, cols)):
        got = ops.column_sum(view).double()
        bound = rows * 2.0 ** -24 * g.double().abs().sum(0) + 1e-30
        assert bool(((got - g.double().sum(0)).abs() <= bound).all())
        ints = (view * 8).round()  # integers: every sum is exact
        assert torch.equal(ops.column_sum(ints).double(), ints.double().sum(0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,k,n", [(1, 48, 5), (17, 1001, 130), (100, 600, 512)])
def test_fused_bias_equals_addition(gpu, tokens, k, n, dtype):
    announce(f"fused bias tokens={tokens} {k}->{n} {dtype}")
    torch.manual_seed(tokens + k)
    layer = t8nn.Linear(k, n, device=gpu).eval()
    layer.bias = torch.nn.Parameter(torch.randn(n, device=gpu, dtype=dtype))
    x = torch.randn((tokens, k), device=gpu, dtype=dtype)
    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    y = layer(a)
    g = torch.randn_like(y)
    y.backward(g)
    db, layer.bias.grad = layer.bias.grad, None
    want = layer.ternary_weight.matmul_input(b) + layer.bias
    want.backward(g)
    assert y.dtype == want.dtype and torch.equal(y, want)
    assert a.grad.dtype == b.grad.dtype and torch.equal(a.grad, b.grad)
    assert db.dtype == layer.bias.grad.dtype
    bound = {torch.float32: tokens * 2.0 ** -23, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -9}
    mags = g.double().abs().sum(0) + 1e-30
    assert bool(((db.double() - layer.bias.grad.double()).abs() <= bound[dtype] * mags).all())


def test_expanded_gradient_and_frozen_input(gpu):
    announce("expanded gradient")
    layer = t8nn.Linear(96, 40, device=gpu).eval()
    x = torch.randn((9, 96), device=gpu, requires_grad=True)
    layer(x).sum().backward()  # an expanded gradient
    t = layer.ternary_weight.trits().float()
    assert torch.equal(x.grad, t.sum(0).expand(9, -1))
    assert torch.equal(layer.bias.grad, torch.full((40,), 9.0, device=gpu))
    layer.bias.grad = None
    layer(x.detach()).sum().backward()  # only the bias needs a gradient
    assert torch.equal(layer.bias.grad, torch.full((40,), 9.0, device=gpu))
    with pytest.raises(ValueError, match="rhs dimension"):
        tensor._linear_under_grad(layer.ternary_weight, torch.randn((2, 95), device=gpu), layer.bias)
