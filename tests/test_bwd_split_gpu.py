"""GPU tests of the split-operand backward (hipgpt_amd/csrc/bwd_half.h) at the
edges of its range: gradients and operands at very different scales, first
tiles that are zero or far smaller than what follows, infinities and NaN, over
head dims (exact, padded, split over waves), ragged lengths, both block sizes,
stored probs and recompute mode; against float64.

Bar, elementwise, from the same sums with absolute values: each product is off
by at most 2^-21 of its size (two fp16 terms each way), dS takes three of them
in turn, and sums over S add 6 S / 16 roundings of 2^-24; in recompute mode P
is off by D 2^-24 of the largest score.  A staged value is held to 2^-32 of its
first tile's largest, so |x| counts as |x| + 2^-11 max |x|, and dS to 2^-34 of
the largest |dO| times the largest |V|.
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


def ref(x, go, p, rel):
    """float64 gradients and their bars."""
    q, k, v, g = x[0].double(), x[1].double(), x[2].double(), go.double()
    c = x.shape[-1] ** -0.5
    dp = torch.matmul(g, v.transpose(-1, -2))
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * c
    want = torch.stack([torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2), q), torch.matmul(p.transpose(-1, -2), g)])

    def up(t):
        return t.abs() + 2.0 ** -11 * t.abs().amax((-1, -2), keepdim=True)

    aq, ak, av, ag = up(q), up(k), up(v), up(g)
    adp = torch.matmul(ag, av.transpose(-1, -2))
    top = g.abs().amax((-1, -2), keepdim=True) * v.abs().amax((-1, -2), keepdim=True)
    ads = (p * (adp + (p * adp).sum(-1, keepdim=True)) + 2.0 ** -14 * top * (p > 0)) * c
    bar = torch.stack([torch.matmul(ads, ak), torch.matmul(ads.transpose(-1, -2), aq),
                       torch.matmul((p + 2.0 ** -18 * (p > 0)).transpose(-1, -2), ag)])
    return want, bar * rel


def check(x, go, causal, recompute, tag):
    S, D = x.shape[-2:]
    s = scores(x, causal)
    p32 = torch.softmax(s, -1).float()
    rel = 3 * 2.0 ** -21 + 6 * S / 16 * 2.0 ** -24
    if recompute:
        rel += D * 2.0 ** -24 * float(s[s > -1e300].abs().max()) * 1.4427
    want, bar = ref(x, go, torch.softmax(s, -1) if recompute else p32.double(), rel)
    got = run(x, go, None if recompute else p32, causal)
    worst = float(((got - want).abs() / bar.clamp_min(1e-300)).max())
    print(tag, tuple(x.shape), causal, recompute, "%.3f of the bar" % worst, flush=True)
    assert ((got - want).abs() <= bar + 1e-36).all()


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("causal", [False, True])
def test_scales(shape, recompute, causal):
    x, go = make(*shape, seed=1)
    check(x, go, causal, recompute, "plain")
    if shape[0] > 8:
        return
    S = shape[2]
    for sq, sk, sv, sg in ((1, 1, 1, 1e-7), (1, 1, 1e-5, 1e3), (8, 1, 300, 1e-2), (1e-4, 1e3, 1, 1e-20), (1, 1, 1e12, 1e-12)):
        y = x * torch.tensor([sq, sk, sv], dtype=torch.float32).view(3, 1, 1, 1, 1)
        check(y, go * sg, causal, recompute, "scales %g %g %g %g" % (sq, sk, sv, sg))
    g = go * torch.exp2(-40.0 * torch.rand(S, 1, generator=torch.Generator().manual_seed(2)))
    check(x, g, causal, recompute, "rows of dO of all sizes")
    g = go.clone()
    g[:, :, : S // 2] = 0  # no loss on the first half
    check(x, g, causal, recompute, "first dO zero")
    y = x.clone()
    y[2, :, :, :40] = 0
    y[1, :, :, :33] = 0
    check(y, go, causal, recompute, "first K, V zero")
    y = x.clone()
    y[:, :, :, S // 2] *= 40.0
    y[2, :, :, S - 1] *= 1e4  # outgrows the first tile's scale
    check(y, go, causal, recompute, "late large rows")


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
