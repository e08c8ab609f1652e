"""GPU tests of the backward on operands split into three bf16 terms
(hipgpt_amd/csrc/terms.h, bwd_terms.h): every operand bit is kept whatever the
other values are, so operands and gradients come at scales far apart, with
features, rows and columns of other sizes, first tiles that are zero, far
smaller or far larger than what follows, very negative scores beside ragged
lengths, infinities and NaN; over head dims (exact, padded, split over waves),
both block sizes, stored probs and recompute mode; against float64.

Bars, element by element, from the same sums with absolute values (e = 2^-24):
a product is off by e of its size and a sum of n of them takes 12 n / 16
roundings; in recompute mode P is off, relatively, by ln 2 times what its score
is (see test_split_range_gpu.py: products, roundings of the sum, of the
exponent and of lse) plus 2^-22 of v_exp_f32, lse by the sum of a row's
exponentials, and O, through the row dots, by the same.  dS = P (dP - Dq) is off by
those shares of P (|dO||V| + sum P |dO||V|).
"""
import numpy as np
import pytest
import torch

from hipgpt_amd import attention as A

pytestmark = pytest.mark.gpu

# (B, H, S, D)
SHAPES = [(1, 3, 300, 32), (2, 2, 261, 64), (1, 2, 333, 128), (2, 3, 75, 48), (1, 2, 130, 96), (3, 2, 31, 20),
          (70, 4, 257, 64), (65, 4, 130, 128)]


def make(B, H, S, D, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(3, B, H, S, D, generator=g), torch.randn(B, H, S, D, generator=g)


def planar(x):
    """[..., B, H, S, D] -> flat rows of tokens"""
    return x.transpose(-2, -3).contiguous().reshape(-1).cuda()


def run(x, go, probs, causal):
    _, B, H, S, D = x.shape
    E = H * D
    grad = torch.full((3 * B * S * E,), 7.0, device="cuda")
    if probs is not None:
        A.attention_backward(planar(go), planar(x), probs.cuda().contiguous(), grad, B, S, E, H, causal=causal)
    else:
        qkv, out, lse = planar(x), torch.empty(B * S, E, device="cuda"), torch.empty(B, H, S, device="cuda")
        A.fwd_lse_qkv_planar(qkv, out, lse, B, S, E, H, causal=causal)
        A.bwd_lse_qkv_planar(planar(go), qkv, out, lse, grad, B, S, E, H, causal=causal)
    torch.cuda.synchronize()
    return grad.cpu().reshape(3, B, S, H, D).transpose(2, 3).double()


def scores(x, causal):
    q, k = x[0].double(), x[1].double()
    s = torch.matmul(q, k.transpose(-1, -2)) / np.sqrt(x.shape[-1])
    return s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool).triu(1), float("-inf")) if causal else s


def ref(x, go, p, s, recompute):
    """float64 gradients and their bars."""
    q, k, v, g = x[0].double(), x[1].double(), x[2].double(), go.double()
    S, D = x.shape[-2:]
    c, e = D ** -0.5, 2.0 ** -24

    def t(m):
        return m.transpose(-1, -2).contiguous()

    dp = torch.matmul(g, t(v))
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * c
    want = torch.stack([torch.matmul(ds, k), torch.matmul(t(ds), q), torch.matmul(t(p), g)])
    n = 2 + 12 * S / 16
    rel = torch.zeros_like(p)
    if recompute:
        live = p > 2.0 ** -60
        mag = torch.matmul(q.abs(), t(k.abs())) * (1.4427 * c)
        smax = torch.where(live, s.abs() * 1.4427, 0.0).amax(-1, keepdim=True)
        rel = (mag * (2 + 12 * D / 16) + 2 * torch.where(p > 0, s.abs(), 0.0) * 1.4427) * e * 0.6932 + 2.0 ** -22
        rel = rel + torch.where(live, rel, 0.0).amax(-1, keepdim=True) + 3 * (smax + np.log2(S) + S) * e
    adp = torch.matmul(g.abs(), t(v.abs()))
    ads = p * (adp + (p * adp).sum(-1, keepdim=True)) * c
    ads = ads * (2 * rel + rel.amax(-1, keepdim=True).clamp_max(1) + (8 + 12 * D / 16 + 2 * n + S / 2) * e)
    apv = p * (rel + n * e)
    bar = torch.stack([torch.matmul(ads, k.abs()), torch.matmul(t(ads), q.abs()), torch.matmul(t(apv), g.abs())])
    # exponentials below fp32's smallest normal are 0
    low = 2.0 ** -126 * S * torch.stack([adp.amax() * k.abs().amax(), adp.amax() * q.abs().amax(), g.abs().amax()])
    return want, bar + (low.view(3, 1, 1, 1, 1) if recompute else 0)


def check(x, go, causal, recompute, tag):
    s = scores(x, causal)
    p32 = torch.softmax(s, -1).float()
    want, bar = ref(x, go, torch.softmax(s, -1) if recompute else p32.double(), s, recompute)
    got = run(x, go, None if recompute else p32, causal)
    worst = float(((got - want).abs() / bar.clamp_min(1e-300)).max())
    print(tag, tuple(x.shape), causal, recompute, "%.3f of the bar" % worst, flush=True)
    assert ((got - want).abs() <= bar + 1e-44).all()


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("causal", [False, True])
def test_scales(shape, recompute, causal):
    x, go = make(*shape, seed=1)
    check(x, go, causal, recompute, "plain")
    if shape[0] > 8:
        return
    S = shape[2]
    for sq, sk, sv, sg in ((1, 1, 1, 1e-7), (1, 1, 1e-5, 1e3), (8, 1, 300, 1e-2), (1e-4, 1e3, 1, 1e-20), (1, 1, 1e12, 1e-12),
                           (1, 1, 1, 1e-30), (1, 1, 1e-30, 1e20)):
        y = x * torch.tensor([sq, sk, sv], dtype=torch.float32).view(3, 1, 1, 1, 1)
        check(y, go * sg, causal, recompute, "scales %g %g %g %g" % (sq, sk, sv, sg))
    g = go * torch.exp2(-40.0 * torch.rand(S, 1, generator=torch.Generator().manual_seed(2)))
    check(x, g, causal, recompute, "rows of dO of all sizes")
    g = go.clone()
    g[:, :, : S // 2] = 0  # no loss on the first half
    check(x, g, causal, recompute, "first dO zero")
    for r in (2.0 ** 18, 2.0 ** 22):
        y = x.clone()
        y[0, ..., 0] *= r  # a feature large in Q and small in K, and the other way round
        y[1, ..., 0] /= r
        y[1, ..., 1] *= r
        y[0, ..., 1] /= r
        check(y, go, causal, recompute, "features times %g" % r)
        y, g = x.clone(), go.clone()
        y[2, ..., 0] *= r
        g[..., 0] /= r
        y[2, ..., 1] /= r
        check(y, g, causal, recompute, "columns of V times %g" % r)
    y = x.clone()
    y[2, :, :, :40] = 0
    y[1, :, :, :33] = 0
    check(y, go, causal, recompute, "first K, V zero")
    for r in (1e-8, 1e4):
        y, g = x.clone(), go.clone()
        y[2, :, :, :32] *= r  # first tiles far from what follows
        g[:, :, :32] *= r
        check(y, g, causal, recompute, "first dO, V times %g" % r)
    y = x.clone()
    y[:, :, :, S // 2] *= 40.0
    y[2, :, :, S - 1] *= 1e4
    check(y, go, causal, recompute, "late large rows")
    y = x.clone()
    y[0] = y[0].abs() * 6  # scores of about -100 and below: exp(-lse) of a key past the last row is infinite
    y[1] = -y[1].abs() * 6
    check(y, go, causal, recompute, "negative scores")


@pytest.mark.parametrize("shape", SHAPES[:6], ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_not_finite(shape, recompute, value):
    """One such entry of dO: its row of dQ and everything of dK and dV that the
    row reaches is not finite (its column of dV, all of dK); other rows of dQ,
    columns of dV and (batch, head) pairs are as without it."""
    B, H, S, D = shape
    x, go = make(*shape, seed=3)
    clean = run(x, go, None if recompute else torch.softmax(scores(x, False), -1).float(), False)
    go[B - 1, H - 1, S // 2, D - 1] = value
    got = run(x, go, None if recompute else torch.softmax(scores(x, False), -1).float(), False)
    ok = torch.ones_like(got, dtype=torch.bool)
    ok[0, B - 1, H - 1, S // 2] = False
    ok[1, B - 1, H - 1] = False
    ok[2, B - 1, H - 1, :, D - 1] = False
    assert not torch.isfinite(got[~ok]).any()
    assert float((got[ok] - clean[ok]).abs().max()) <= 1e-5 * float(clean.abs().max())
