"""The training kernels of t8.nn.Linear (csrc/qat.hip, the three-plane product) against the
tensor expression they stand in for, F.linear(x, ternary(w / s) * s, b).

Scale, ternarized weight and the weight gradient's passes keep the expression's roundings, so
they are compared bit for bit (NaN as NaN), in each weight type, at the edges of a
12-weight run, of a limb and of the thresholds.  The products sum in float32 in another
order: with K terms both sides are within (K + 2) 2^-24 sum |x q s| of the exact value
(products of the three planes are exact; the expression rounds each product once more; bit
for bit, in every plane: test_gpu_plane_pairs.py),
doubled for the matrix cores' own rounding.
"""

from __future__ import annotations

import pytest
import torch
from torch.nn import functional as F

from t81lib_amd import nn as t8nn
from t81lib_amd import qat
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24


def same_bits(a, b, what):
    a, b = a.detach(), b.detach()
    assert a.shape == b.shape and a.dtype == b.dtype, what
    eq = (a == b) | (a.isnan() & b.isnan())
    assert bool(eq.all()), f"{what}: {int((~eq).sum())} of {a.numel()} differ"


def expression(weight, scale, threshold):
    return qat.ternary(weight / scale, threshold=threshold) * scale


def expression_scale(weight, existing):
    candidate = weight.detach().abs().amax().clamp(min=1e-6).to(torch.float32)
    if existing is None:
        return candidate
    return (existing.to(torch.float32) * 0.99 + candidate * 0.01).clamp(min=1e-6)


def edge_weight(rows, cols, dtype, gpu, threshold, special=True):
    g = torch.Generator("cpu").manual_seed(rows * 7 + cols)
    w = torch.randn((rows, cols), generator=g) * 0.02
    flat = w.view(-1)
    s = float(w.abs().max())
    marks = [threshold * s, -threshold * s, 0.5 * s, -0.5 * s, s, -s, 0.0, -0.0, 1e-30]
    near = []
    for m in marks:
        t = torch.tensor(m, dtype=torch.float32)
        near += [m, float(torch.nextafter(t, torch.tensor(1.0))),
                 float(torch.nextafter(t, torch.tensor(-1.0)))]
    near = [v for v in near if abs(v) <= s][:flat.numel()]
    flat[:len(near)] = torch.tensor(near)
    return w.to(dtype).to(gpu)


SHAPES = [(1, 1), (3, 11), (5, 12), (4, 13), (7, 48), (2, 49), (33, 100), (64, 4096), (130, 1001)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_weight_passes_bit_exact(gpu, rows, cols, dtype):
    announce(f"qat weight {rows}x{cols} {dtype}")
    for threshold in (0.0, 0.45, 0.5, 1.0, 3.0):
        w = edge_weight(rows, cols, dtype, gpu, min(threshold, 1.0))
        scale = existing = None
        for step in range(3):  # first scale, then its moving average
            want = expression_scale(w * (1 + step), existing)
            scale = qat.training_scale(w * (1 + step), existing)
            same_bits(scale, want, f"scale {step}")
            existing = want
        a = w.clone().requires_grad_(True)
        b = w.clone().requires_grad_(True)
        wq, packed = qat.TernaryWeight.apply(a, scale, threshold)
        want = expression(b, scale, threshold)
        same_bits(wq, want, f"weight thr={threshold}")
        g = torch.randn((rows, cols), device=gpu).to(dtype)
        wq.backward(g)
        want.backward(g)
        same_bits(a.grad, b.grad, f"gradient thr={threshold}")


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 0.0])
def test_weight_passes_non_finite_and_zero(gpu, value):
    announce(f"qat weight with {value}")
    w = torch.zeros((6, 50), device=gpu) if value == 0.0 else edge_weight(6, 50, torch.float32, gpu, 0.45)
    w[2, 17] = value
    scale = qat.training_scale(w, None)
    same_bits(scale, expression_scale(w, None), "scale")
    a, b = w.clone().requires_grad_(True), w.clone().requires_grad_(True)
    wq, _ = qat.TernaryWeight.apply(a, scale, 0.45)
    want = expression(b, scale, 0.45)
    same_bits(wq, want, "weight")
    g = torch.randn_like(w)
    wq.backward(g)
    want.backward(g)
    same_bits(a.grad, b.grad, "gradient")


def layers(n, k, bias, gpu):
    layer = t8nn.Linear(k, n, bias=bias, device=gpu)
    with torch.no_grad():
        layer.weight.normal_(0.0, 0.02)
    return layer.train()


# M, K, N: one pair of limbs, odd limb counts, K % 8 != 0, a token past a block, split K
STEPS = [(65, 40, 24), (70, 97, 513), (100, 1001, 300), (257, 4096, 512), (96, 6000, 130)]


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("M,K,N", STEPS)
def test_training_step(gpu, monkeypatch, M, K, N, bias):
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0 if K % 2 == 0 else 1 << 40)
    announce(f"qat step M={M} K={K} N={N} bias={bias}")
    torch.manual_seed(M + K + N)
    layer = layers(N, K, bias, gpu)
    x = torch.randn((2, M // 2, K) if M % 2 == 0 else (M, K), device=gpu).requires_grad_(True)
    assert qat.product_on_kernels(x, layer.weight, layer.bias)
    y = layer(x)
    g = torch.randn_like(y)
    y.backward(g)
    s = expression_scale(layer.weight, None)
    same_bits(layer.training_scale, s, "scale")
    wq = expression(layer.weight.detach(), s, 0.45).double()
    x2, g2 = x.detach().reshape(-1, K).double(), g.reshape(-1, N).double()

    def close(got, want, terms, mags, what):
        bound = 2.0 * (terms + 2) * U32 * mags + 1e-30
        err = (got.detach().reshape(want.shape).double() - want).abs()
        assert bool((err <= bound).all()), f"{what}: {float((err / bound).max())} of the bound"

    b = layer.bias.detach().double() if bias else torch.zeros(N, device=gpu, dtype=torch.float64)
    close(y, x2 @ wq.T + b, K, x2.abs() @ wq.abs().T + b.abs(), "y")
    close(x.grad, g2 @ wq, N, g2.abs() @ wq.abs(), "dx")
    u = layer.weight.detach() / s
    close(layer.weight.grad, torch.where(u.abs() < 0.5, 2.0 * (g2.T @ x2), torch.zeros_like(wq)),
          6 * M + 4, 2.0 * (g2.abs().T @ x2.abs()), "dw")
    if bias:
        close(layer.bias.grad, g2.sum(0), M, g2.abs().sum(0), "db")


def test_training_second_derivative_and_stale_graph(gpu, monkeypatch):
    """create_graph builds the expression's graph; a graph outlives a change of the weight."""
    announce("qat second derivative")
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    torch.manual_seed(5)
    M, K, N = 80, 60, 36
    layer = layers(N, K, True, gpu)
    x = torch.randn((M, K), device=gpu).requires_grad_(True)

    def second(f):
        x.grad = layer.weight.grad = None
        (gx,) = torch.autograd.grad(f().square().sum(), x, create_graph=True)
        gx.square().sum().backward()
        return gx.detach(), x.grad, layer.weight.grad

    got = second(lambda: layer(x))
    s = layer.training_scale
    want = second(lambda: F.linear(x, expression(layer.weight, s, 0.45), layer.bias))
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.abs().max()))
    y = layer(x)
    with torch.no_grad():
        layer.weight.add_(1.0)
    y.sum().backward()  # the graph keeps what it needs of the old weight


def test_training_routes(gpu, monkeypatch):
    """Small products, autocast, other types, strides and forward-mode keep F.linear."""
    announce("qat routes")
    layer = layers(40, 48, True, gpu)
    x = torch.randn((80, 48), device=gpu)
    assert not qat.product_on_kernels(x, layer.weight, layer.bias)
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    assert qat.product_on_kernels(x, layer.weight, layer.bias)
    assert not qat.product_on_kernels(x[:0], layer.weight, layer.bias)
    assert not qat.product_on_kernels(x.t().contiguous().t(), layer.weight, layer.bias)
    assert not qat.product_on_kernels(x.bfloat16(), layer.weight, layer.bias)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not qat.product_on_kernels(x, layer.weight, layer.bias)
        assert layer(x).dtype == torch.bfloat16
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        y = layer(dual)
        assert torch.autograd.forward_ad.unpack_dual(y).tangent is not None
    torch.manual_seed(1)
    layer.configure_qat(stochastic_rounding=True)
    a = layer(x)
    torch.manual_seed(1)
    assert torch.equal(a, F.linear(x, layer._quantize_training_weight(), layer.bias))


# M, N, K: one row, a row past a step of 16, columns past a block of 32 and a tile of 256, K that
# takes no 16-byte stores, the tokens split (few tiles), odd and even step counts
PRODUCTS = [(1, 1, 1), (17, 33, 40), (32, 256, 32), (100, 257, 300), (1000, 511, 1025),
            (260, 1030, 258), (1040, 130, 64)]


@pytest.mark.parametrize("M,N,K", PRODUCTS)
def test_weight_product(gpu, monkeypatch, M, N, K):
    """Six plane products of M exact terms each, summed in float32: within 2 (6 M + 4) 2^-24
    sum |g x| (doubled for the matrix cores' rounding); the plane products left out are below
    2^-24 of each term, inside the + 4.  Infinities and NaN as the float32 product gives them.
    (Bit for bit, in every pair of planes: test_gpu_plane_pairs.py.)"""
    announce(f"qat weight product M={M} N={N} K={K}")
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    gen = torch.Generator("cpu").manual_seed(M + N + K)
    g = torch.randn((M, N), generator=gen).to(gpu)
    x = (torch.randn((M, K), generator=gen) * 10.0 ** torch.randint(-3, 4, (M, 1), generator=gen)).to(gpu)
    want, mags = g.double().T @ x.double(), g.double().abs().T @ x.double().abs()
    err = (qat.weight_product(g, x).double() - want).abs()
    assert bool((err <= 2.0 * (6 * M + 4) * U32 * mags + 1e-30).all())
    ints = torch.randint(-100, 101, (M, N), generator=gen).float().to(gpu)
    xi = torch.randint(-100, 101, (M, K), generator=gen).float().to(gpu)  # exact sums
    assert torch.equal(qat.weight_product(ints, xi).double(), ints.double().T @ xi.double())
    g[M // 2, N // 3] = float("inf")
    x[M - 1, K // 2] = float("-inf")
    x[0, 0] = float("nan")
    got = qat.weight_product(g, x)
    # of an infinity's products with finite values, all but those with zeros are infinities
    ref = g.double().T @ x.double()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert bool(((got.double() - ref).abs()[ok] <= 2.0 * (6 * M + 4) * U32 * mags[ok] + 1e-30).all())
    top = torch.full((M, K), 3.4e38, device=gpu)  # finite, past bf16's largest value
    assert bool(qat.weight_product(torch.full((M, N), 1e-3 / M, device=gpu), top).isfinite().all())


def test_dispatch_modes(gpu, monkeypatch):
    """Under a dispatch mode (make_fx) the expression runs, so that its operations are seen."""
    announce("qat dispatch modes")
    from torch.fx.experimental.proxy_tensor import make_fx

    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    layer = layers(40, 48, True, gpu)
    x = torch.randn((6, 48), device=gpu)
    want = F.linear(x, expression(layer.weight, expression_scale(layer.weight, None),
                                  layer.ternary_threshold), layer.bias)
    with torch.no_grad():
        traced = make_fx(lambda v: layer(v))(x)
        layer.training_scale = None
        assert torch.allclose(traced(x), want, rtol=1e-5, atol=1e-5)
    assert any(s in str(n.target) for n in traced.graph.nodes for s in ("mm", "linear"))


def test_saved_tensors_of_another_type(gpu, monkeypatch):
    """Hooks that return another type than was saved: the weight gradient's map by its values, a
    product of mixed types refused as torch refuses it."""
    announce("qat saved-tensor hooks")
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    layer = layers(40, 48, True, gpu)
    x = torch.randn((80, 48), device=gpu)
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: t, lambda t: t.to(torch.int32) if t.dtype == torch.uint16 else t):
        layer(x).sum().backward()
    got = layer.weight.grad.clone()
    layer.weight.grad = None
    layer.training_scale = None
    layer(x).sum().backward()
    assert torch.allclose(got, layer.weight.grad, rtol=1e-5, atol=1e-6)
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: t, lambda t: t.bfloat16() if t.shape == x.shape else t):
        out = layer(x).sum()
    with pytest.raises(RuntimeError):
        out.backward()


def test_scale_of_other_shapes(gpu, monkeypatch):
    """A training scale that a program set to more than one value keeps the expression's
    broadcast (and, for bfloat16 weights, its float32 result): the kernels read one value."""
    announce("qat scales per row")
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    for dtype, shape in [(torch.float32, (40, 1)), (torch.float32, (48,)), (torch.bfloat16, (1,))]:
        layer = layers(40, 48, False, gpu).to(dtype)
        x = torch.randn((80, 48), device=gpu)
        start = torch.rand(shape, device=gpu) * 0.1 + 0.02
        layer.training_scale = start
        want = F.linear(x, expression(layer.weight, expression_scale(layer.weight, start),
                                      layer.ternary_threshold))
        assert torch.equal(layer(x), want)
        assert torch.equal(layer.training_scale, expression_scale(layer.weight, start))

    class PerRow(t8nn.Linear):
        def _update_training_scale(self):
            return self.weight.detach().abs().amax(1, keepdim=True)

    layer = PerRow(48, 40, bias=False, device=gpu).train()
    scale = layer._update_training_scale()
    assert torch.equal(layer(x), F.linear(x, expression(layer.weight, scale,
                                                        layer.ternary_threshold)))
