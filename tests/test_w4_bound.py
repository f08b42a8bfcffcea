"""CPU: the limits that the W4 head's GPU test holds it to let float32 sums in the kernels' order through
and refuse a reference with a small mistake."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from w4_bound import w4_limits   # noqa: E402

M, N = 48, 256


@pytest.fixture(params=[128, 640, 2560, 4096])
def head(request):
    """x, codes, scale, zero of the GPU test's distributions, float64 (scale and zero [N, G, 1])."""
    K = request.param
    gen = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=gen).bfloat16().double()
    q = torch.randint(0, 16, (N, K // 128, 128), generator=gen).double()
    scale = (torch.rand(N, K // 128, 1, generator=gen) * 0.01 + 1e-3).bfloat16().double()
    zero = torch.randint(-20, 36, scale.shape, generator=gen).double()
    return x, q, scale, zero


def weight(q, scale, zero):
    return ((q - zero) * scale).flatten(1)


def limits(x, q, scale, zero):
    return w4_limits(x, weight(q, scale, zero), ((q + 256 + zero.abs()) * scale).flatten(1))


def outside(y, lim):
    y = y.bfloat16().double()
    return ((y < lim[0]) | (y > lim[1])).double().mean(0)      # share of the rows, per output


@pytest.mark.parametrize("order", ["sequential", "truncated"])
def test_float32_sums_are_inside(head, order):
    """Group products of x with 128 + code and of the offset, product by product in float32 (or, as an
    accumulator without rounding might, each sum cut off toward zero), then the groups."""
    x, q, scale, zero = head
    add = lambda a, b: a + b
    if order == "truncated":
        def add(a, b):
            s = a.double() + b.double()
            f = s.float()
            return torch.where(f.double().abs() > s.abs(), torch.nextafter(f, f.new_zeros(())), f)
    acc = torch.zeros(M, N)
    for g in range(q.shape[1]):
        d, n = torch.zeros(M, N), torch.zeros(M, 1)
        for j in range(128):
            xj = x[:, g * 128 + j].float()
            d = add(d, xj[:, None] * (128 + q[:, g, j].float())[None])
            n = add(n, -xj[:, None])
        s, z = scale[:, g, 0], zero[:, g, 0]
        t = (n.double() * (128 + z) + d.double()).float()
        acc = (s * t.double() + acc.double()).float()
    assert outside(acc, limits(x, q, scale, zero)).max() == 0


def test_mistakes_are_outside(head):
    x, q, scale, zero = head
    lim = limits(x, q, scale, zero)
    assert outside(x @ weight(q, scale, zero).T, lim).max() == 0
    off = zero.clone()
    off[:, -1] += 1                                  # one group's zero point off by one
    assert outside(x @ weight(q, scale, off).T, lim).mean() > 0.4
    w = weight(q, scale, zero)
    w[:, -8:] = 0                                    # eight products left out
    assert outside(x @ w.T, lim).mean() > 0.8
    one = q.clone()
    one[:, 0, 5] = (one[:, 0, 5] + 8) % 16           # one code of a row
    assert outside(x @ weight(one, scale, zero).T, lim).max(0).values > 0.3
