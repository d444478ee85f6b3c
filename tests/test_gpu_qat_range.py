"""The training products where float32 overflows: as a float32 product gives them.

The products run as sums over bf16 planes, which must not overflow where the float32 sum does
not (a hi plane rounds up, and a training scale below one is applied after the sum), and must
come out as the infinity, never as infinity - infinity, where it does.
"""

from __future__ import annotations

import pytest
import torch

from t81lib_amd import ops, qat
from test_gpu_exact_f32 import announce
from test_gpu_qat import PRODUCTS, U32, expression, expression_scale, layers

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


@pytest.mark.parametrize("M,N,K", PRODUCTS)
def test_weight_product_small_values(gpu, monkeypatch, M, N, K):
    """Every float32 value is held to its last bit, subnormal ones too: one term per output, so
    the product is exact."""
    announce(f"qat weight product small values M={M} N={N} K={K}")
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    gen = torch.Generator("cpu").manual_seed(M + N * 3 + K)
    exps = torch.randint(-149, -90, (M, K), generator=gen).double()
    x = (torch.randint(1, 1 << 24, (M, K), generator=gen).double() * 2.0 ** exps).float().to(gpu)
    one = torch.zeros((M, N))
    one[torch.randint(0, M, (N,), generator=gen), torch.arange(N)] = 1.0
    for g, v in ((one.to(gpu), x), (x, one.to(gpu))):
        got, want = qat.weight_product(g, v), g.double().T @ v.double()
        assert torch.equal(got.double(), want)


@pytest.mark.parametrize("M,K,N", [(70, 97, 513), (100, 1001, 300), (96, 6000, 130)])
def test_training_product_small_and_large_values(gpu, M, K, N):
    """One term per output: values whose digits end at 2^-140 or above, up to the largest, are
    held to the last bit."""
    announce(f"qat product small values M={M} K={K} N={N}")
    gen = torch.Generator("cpu").manual_seed(M + N * 3 + K)
    exps = torch.where(torch.rand((M, K), generator=gen) < 0.5,
                       torch.randint(-140, -100, (M, K), generator=gen),
                       torch.randint(60, 105, (M, K), generator=gen)).double()
    x = (torch.randint(1, 1 << 24, (M, K), generator=gen).double() * 2.0 ** exps).float()
    x[:, 0], x[:, 1] = 3.4028234e38, -3.3953138e38  # the largest float32, and past bf16's
    t = torch.zeros((N, K))
    at = torch.randint(0, K, (N,), generator=gen)
    at[0], at[1] = 0, 1
    t[torch.arange(N), at] = 1.0
    x, packed = x.to(gpu), ops.quantize_pack(t.to(gpu), 0.5)
    for s in (1.0, 0.5):
        got = qat._matmul(x, packed, N, torch.tensor(s, device=gpu), None)
        want = (s * x.double()[:, at.to(gpu)])
        assert torch.equal(got.double(), want.float().double())


@pytest.mark.parametrize("std", [0.02, 30.0])
@pytest.mark.parametrize("M,K,N", [(70, 97, 513), (100, 1001, 300), (96, 6000, 130)])
def test_training_product_overflow(gpu, monkeypatch, M, K, N, std):
    """Activations and gradients near the largest float32: sums that the scaled weights keep in
    range stay finite (each output within the float32 summation bound), others do not become
    NaN."""
    announce(f"qat product overflow M={M} K={K} N={N} std={std}")
    monkeypatch.setattr(qat, "MIN_PRODUCT", 0)
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 1 << 40)
    torch.manual_seed(M + K + N)
    layer = layers(N, K, False, gpu)
    with torch.no_grad():
        layer.weight.mul_(std / 0.02)
    top = 3.0e38 / max(1.0, float(layer.weight.detach().abs().max()))

    # ordinary values, and in half the rows about eight near the top
    def values(rows, cols, scale):
        v = torch.randn((rows, cols), device=gpu)
        big = (torch.rand((rows, 1), device=gpu) < 0.5) & (torch.rand((rows, cols), device=gpu) < 8 / cols)
        return torch.where(big, (0.9 + 0.1 * torch.rand_like(v)) * scale, v)

    x = values(M, K, top).requires_grad_(True)
    y = layer(x)
    g = values(M, N, top)
    y.backward(g)
    s = expression_scale(layer.weight, None)
    wq = expression(layer.weight.detach(), s, 0.45).double()
    for got, a, b in ((y, x.detach(), wq.T), (x.grad, g, wq)):
        want, mags = a.double() @ b, a.double().abs() @ b.abs()
        got = got.detach().double()
        sure = mags < 3.4e38  # no order of the sum overflows
        assert bool(sure.any()) and not bool(got[sure].isinf().any())
        assert not bool(got.isnan().any())
        bound = 2.0 * (a.shape[1] + 2) * U32 * mags + 1e-30
        assert bool(((got - want).abs() <= bound)[sure].all())


def test_weight_product_under_graph_capture(gpu, monkeypatch):
    """The note of large values is the launch's own: replays on inputs that turn large and back
    equal the eager results, with eager work between them."""
    announce("qat weight product graph capture")
    monkeypatch.setattr(qat, "MIN_WEIGHTS", 0)
    M, N, K = 1040, 130, 64  # (the tokens split)
    torch.manual_seed(9)
    g, x = torch.randn((M, N), device=gpu), torch.randn((M, K), device=gpu)
    plain = x.clone()
    large = x.clone()
    large[5, 7] = 1e20
    infinite = x.clone()
    infinite[5, 7] = float("inf")
    want = {}
    for name, v in (("plain", plain), ("large", large), ("infinite", infinite)):
        want[name] = qat.weight_product(g, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = qat.weight_product(g, x)
    for name, v in (("large", large), ("plain", plain), ("infinite", infinite), ("plain", plain),
                    ("plain", plain), ("large", large)):
        x.copy_(v)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        same = (out == want[name]) | (out.isnan() & want[name].isnan())
        assert bool(same.all()), name
        other = qat.weight_product(g, infinite)  # eager work in between
        del other
    del graph
