"""Inputs that pin products of three bf16 planes (x = hi + mid + lo) bit for bit, and a proof on
the CPU that they do: leaving any one plane, or any pair of planes, out of a product of them
changes results at every size they are used at.

Values are integers, at most three non-zero terms meet per output, and every partial sum of
plane products, in any order, is an integer below 2^24: a float32 sum of them is exact.
"""

from __future__ import annotations

import itertools

import pytest
import torch

from test_gpu_qat import PRODUCTS, STEPS

PAIRS = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]  # that the weight's gradient sums
LONG = (1 << 22) - (1 << 15)   # 3 terms of 22 bits: all three planes
SHORT = (1 << 11) - 1          # 3 products of 11 by 11 bits: hi and mid of both


def integers(gen, shape, top):
    """Signed integers of top's size, whose planes' digits are seldom zeros."""
    v = torch.randint(top // 2, top + 1, shape, generator=gen) | 1
    return (v * (2 * torch.randint(0, 2, shape, generator=gen) - 1)).float()


def few(gen, rows, cols, top):
    """A rows x cols matrix with three non-zeros per column (one row: one), the last row among
    them in every fourth column and the first in every fourth."""
    out = torch.zeros((rows, cols))
    at = torch.stack([torch.randperm(rows, generator=gen)[:3] for _ in range(cols)], 1)
    at[0, 0::4], at[0, 1::4] = rows - 1, 0
    out.scatter_(0, at, integers(gen, at.shape, top))
    return out


def weight_product_inputs(M, N, K):
    """(G, X) of each kind: short by short, one by long, long by one."""
    gen = torch.Generator("cpu").manual_seed(M + 5 * N + 7 * K)
    yield few(gen, M, N, SHORT), integers(gen, (M, K), SHORT)
    yield few(gen, M, N, 1), integers(gen, (M, K), LONG)
    yield integers(gen, (M, N), LONG), few(gen, M, K, 1)


def ternary_inputs(M, K, N):
    """(X, T) for X T^T with three trits per row of T (as few() has them per column)."""
    gen = torch.Generator("cpu").manual_seed(M + 5 * N + 7 * K)
    return integers(gen, (M, K), LONG), few(gen, K, N, 1).T.contiguous()


def planes(x):
    out = []
    for _ in range(3):
        out.append(x.bfloat16().float())
        x = x - out[-1]
    assert not bool(x.any())
    return [p.double() for p in out]


@pytest.mark.parametrize("M,N,K", PRODUCTS)
def test_each_pair_of_planes_matters(M, N, K):
    missed = set(PAIRS)
    for g, x in weight_product_inputs(M, N, K):
        gp, xp = planes(g), planes(x)
        want = g.double().T @ x.double()
        assert float((sum(p.abs() for p in gp).T @ sum(p.abs() for p in xp)).max()) < 2 ** 24
        terms = {p: gp[p[0]].T @ xp[p[1]] for p in itertools.product(range(3), repeat=2)}
        assert torch.equal(sum(terms[p] for p in PAIRS), want)  # the three left out are zeros
        # a pair counts where leaving it out changes nine outputs of ten
        missed -= {p for p in PAIRS if float((terms[p] != 0).float().mean()) > 0.9}
    assert not missed


@pytest.mark.parametrize("M,K,N", STEPS)
def test_each_plane_matters(M, K, N):
    x, t = ternary_inputs(M, K, N)
    xp, t = planes(x), t.double()
    assert float((sum(p.abs() for p in xp) @ t.abs().T).max()) < 2 ** 24
    for p in xp:
        assert float(((p @ t.T) != 0).float().mean()) > 0.9
