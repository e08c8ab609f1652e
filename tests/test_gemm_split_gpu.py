"""GPU tests of the projection GEMM on operands split into three bf16 terms
(hipgpt_amd/csrc/terms.h, gemm.hip): every operand bit is kept whatever the
other values of its row or column are, so rows, columns and single features
of very different size, tiny and huge values, and rows and columns of zeros
are all held to the error of fp32 sums; infinities, NaN and values past the
terms' range; tile edges.  Against float64.

Bars.  A product is off by at most 2^-24 of its size (the dropped terms), and a
sum over k takes six MFMAs per 16 indices, each adding its products in two
groups: n = 12 K / 16 roundings of 2^-24 of what the sum then is.  Per element
that is at most (1 + n) 2^-24 sum |a||w|; over all elements, as roundings are
independent, its root mean square relative to sqrt(sum a^2 w^2) is at most
(1 + sqrt(n)) 2^-24 (no value enters that is shared with other products).
"""
import numpy as np
import pytest
import torch

from hipgpt_amd import projection as P

pytestmark = pytest.mark.gpu

# each tile shape (by the number of 128 x 128 tiles), edges, K tails
SHAPES = [(1, 4, 4), (70, 132, 36), (130, 260, 100), (257, 128, 32), (64, 256, 768), (2048, 2052, 68), (4100, 1028, 32)]


def inputs(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g), torch.randn(K, N, generator=g), torch.randn(N, generator=g)


def check(a, w, b, tag, ok=None):
    got = P.gemm_bias(a.cuda(), w.cuda(), b.cuda()).cpu().double()
    a64, w64, b64 = a.double(), w.double(), b.double()
    n = 12 * a.shape[1] / 16
    err = (got - (a64 @ w64 + b64)).abs()
    sums = (a64.abs() @ w64.abs()) * 2.0 ** -24
    bias = b64.abs() * 2.0 ** -23 + sums
    bad = ~(err <= sums * (1 + n) + bias + 1e-44)  # 1e-44: fp32's smallest steps
    size = torch.sqrt((a64 ** 2) @ (w64 ** 2)) * 2.0 ** -24
    live = (size > 2.0 ** -140) & torch.isfinite(size)
    if ok is not None:
        bad &= ok  # rows or columns that are not finite are looked at apart
        live &= ok
    rel = float(torch.sqrt((((err - bias).clamp_min(0) / size)[live] ** 2).mean())) if live.any() else 0.0
    print(tag, tuple(a.shape), tuple(w.shape), int(bad.sum()), "%.3f of %.3f" % (rel, 1 + n ** 0.5), flush=True)
    assert not bad.any()
    assert rel <= 1 + n ** 0.5
    return got


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_scales(M, N, K):
    a, w, b = inputs(M, N, K, 1)
    check(a, w, b, "plain")
    sa = torch.exp2(torch.arange(M) % 61 - 30.0).view(M, 1)  # every row and column its own size
    sw = torch.exp2(torch.arange(N) % 41 - 20.0).view(1, N)
    zero = torch.zeros(N)
    check(a * sa, w * sw, zero, "row and column scales")
    z = a.clone()
    z[::2, : min(K, 40)] = 0  # rows that begin with zeros, rows of zeros
    z[::5] = 0
    y = w.clone()
    y[: min(K, 40), ::3] = 0
    y[:, 1::7] = 0
    check(z * 1e-6, y * 1e-5, b, "zeros first")
    z = a.clone()
    z[:, K - 1] *= 1e5
    z[0] *= torch.exp2(torch.arange(K) % 16 - 8.0)
    check(z, w, b, "late large values")
    check(a * 1e25, w * 1e-25, b, "large times small")
    for r in (2.0 ** 14, 2.0 ** 18, 2.0 ** 22, 2.0 ** 40, 2.0 ** -22):  # features of another unit, weights that undo it
        z, y = a.clone(), w.clone()
        z[:, 0] *= r
        y[0] /= r
        check(z, y, zero, "feature times %g" % r)
    for sa, sw in ((1e36, 1e-25), (1e-25, 1e36), (1, 1e-33), (1, 1e-36), (1e-36, 1), (1e10, 1e-36), (1e30, 1e5)):
        check(a * sa, w * sw, zero, "%g times %g" % (sa, sw))


@pytest.mark.parametrize("M,N,K", SHAPES[1:6])
def test_exact(M, N, K):
    """Products by a power of two are exact, so a permutation of scaled unit
    rows returns W bit for bit; and a row does not see the other rows."""
    a, w, b = inputs(M, N, K, 4)
    unit = torch.zeros(M, K)
    rows, cols = torch.arange(M), (torch.arange(M) * 7) % K
    unit[rows, cols] = torch.exp2((torch.arange(M) % 21 - 10).float())
    got = P.gemm_bias(unit.cuda(), w.cuda()).cpu()
    assert torch.equal(got, w[cols] * unit[rows, cols].view(M, 1))
    plain = P.gemm_bias(a.cuda(), w.cuda(), b.cuda()).cpu()
    z = a.clone()
    z[M // 2] *= 1e8
    z[M // 3] = 0
    got = P.gemm_bias(z.cuda(), w.cuda(), b.cuda()).cpu()
    keep = (rows != M // 2) & (rows != M // 3)
    assert torch.equal(got[keep], plain[keep])


@pytest.mark.parametrize("M,N,K", SHAPES[1:6])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38])
def test_not_finite(M, N, K, value):
    a, w, b = inputs(M, N, K, 2)
    m, n = M // 2, N // 3
    w = w * 0.1  # 3e38: past the terms' range, within fp32's
    a[m, K // 2] = value
    ok = torch.ones(M, N, dtype=torch.bool)
    ok[m] = bool(np.isfinite(value))
    got = check(a, w, b, "A " + str(value), ok)
    want = torch.sign(w[K // 2]) * value
    if not np.isfinite(value):
        assert torch.isnan(got[m]).all() if np.isnan(value) else (got[m] == want.double()).all()
    a, w, b = inputs(M, N, K, 3)
    a = a * 0.1
    w[K - 1, n] = value
    ok = torch.ones(M, N, dtype=torch.bool)
    ok[:, n] = bool(np.isfinite(value))
    got = check(a, w, b, "W " + str(value), ok)
    want = torch.sign(a[:, K - 1]) * value
    if not np.isfinite(value):
        assert torch.isnan(got[:, n]).all() if np.isnan(value) else (got[:, n] == want.double()).all()
