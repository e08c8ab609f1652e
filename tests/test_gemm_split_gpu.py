"""GPU tests of the projection GEMM on split operands (hipgpt_amd/csrc/gemm.hip):
rows of A and columns of W of very different size, rows and columns that begin
with (or are all) zeros, values that outgrow the scale their first k-tile gave
them, infinities and NaN, and tile edges, against float64.

Bar per element: the sum over k of |a||w| times 2^-21 (two fp16 terms hold 2^-22
of a product each way), plus 2^-24 of the same sum for each addition (16 indices
take three MFMAs, each of which adds its products in two groups: 6 K / 16),
plus the terms' absolute floor: with a row's first k-tile scaled to at most 2^8
and fp16 steps of 2^-24, a value is off by up to 2^-32 of the row's largest
magnitude (a column's likewise).
"""
import numpy as np
import pytest
import torch

from hipgpt_amd import projection as P

pytestmark = pytest.mark.gpu

# both tile shapes (fewer and more than 256 tiles of 128 x 128), edges, K tails
SHAPES = [(1, 4, 4), (70, 132, 36), (130, 260, 100), (257, 128, 32), (2048, 2052, 68), (4100, 1028, 32)]


def inputs(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g), torch.randn(K, N, generator=g), torch.randn(N, generator=g)


def check(a, w, b, tag, ok=None):
    got = P.gemm_bias(a.cuda(), w.cuda(), b.cuda()).cpu().double()
    want = a.double() @ w.double() + b.double()
    K = a.shape[1]
    aa, ww = a.double().abs(), w.double().abs()
    floor = aa.amax(1, keepdim=True) * ww.sum(0, keepdim=True) + aa.sum(1, keepdim=True) * ww.amax(0, keepdim=True)
    bar = (aa @ ww) * (2.0 ** -21 + 6 * K / 16 * 2.0 ** -24) + floor * 2.0 ** -32 + b.abs() * 2.0 ** -23 + 1e-37
    bad = ~((got - want).abs() <= bar)
    if ok is not None:
        bad &= ok  # rows or columns that are not finite are looked at apart
    print(tag, tuple(a.shape), tuple(w.shape), int(bad.sum()), flush=True)
    assert not bad.any()
    return got


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_scales(M, N, K):
    a, w, b = inputs(M, N, K, 1)
    check(a, w, b, "plain")
    sa = torch.exp2(torch.arange(M) % 61 - 30.0).view(M, 1)  # every row and column its own size
    sw = torch.exp2(torch.arange(N) % 41 - 20.0).view(1, N)
    check(a * sa, w * sw, torch.zeros(N), "row and column scales")
    z = a.clone()
    z[::2, : min(K, 40)] = 0  # rows that begin with zeros, rows of zeros
    z[::5] = 0
    y = w.clone()
    y[: min(K, 40), ::3] = 0
    y[:, 1::7] = 0
    check(z * 1e-6, y * 1e-5, b, "zeros first")
    z = a.clone()
    z[:, K - 1] *= 1e5  # outgrows the first k-tile's scale
    z[0] *= torch.exp2(torch.arange(K) % 16 - 8.0)
    check(z, w, b, "late large values")
    check(a * 1e25, w * 1e-25, b, "large times small")


@pytest.mark.parametrize("M,N,K", SHAPES[1:5])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_not_finite(M, N, K, value):
    a, w, b = inputs(M, N, K, 2)
    m, n = M // 2, N // 3
    a[m, K // 2] = value
    ok = torch.ones(M, N, dtype=torch.bool)
    ok[m] = False
    got = check(a, w, b, "A " + str(value), ok)
    want = torch.sign(w[K // 2]) * value
    assert torch.isnan(got[m]).all() if np.isnan(value) else (got[m] == want.double()).all()
    a, w, b = inputs(M, N, K, 3)
    w[K - 1, n] = value
    ok = torch.ones(M, N, dtype=torch.bool)
    ok[:, n] = False
    got = check(a, w, b, "W " + str(value), ok)
    want = torch.sign(a[:, K - 1]) * value
    assert torch.isnan(got[:, n]).all() if np.isnan(value) else (got[:, n] == want.double()).all()
