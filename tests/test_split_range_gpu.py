"""GPU tests of the fp32 forward on operands split into three bf16 terms
(hipgpt_amd/csrc/terms.h): every operand bit is kept whatever the other values
are, so Q, K and V come at scales far apart, with single outliers, single tiny
or huge columns, rows and features, and with infinities, NaN and values past
the terms' range (whose workgroups run again on fp32 MFMA), in each workgroup
shape of the dispatch and at ragged sizes.

Finite cases against float64, element by element and relative to what the
element itself is made of.  A score (log2 units) is a D-term sum of magnitude
abs = sum |q||k|: its products are each off by 2^-24 of their size, and six
MFMAs per 16 dims add them in two groups, 12 D / 16 roundings of 2^-24 abs; the
exponent's own rounding (|s| 2^-24) and that of v_exp_f32 (2^-22) come on top.
An exponential is off by that times ln 2, relatively, and so is the row's sum,
which adds up to Sk / 2 of them in one chain; P takes its logarithm into the
exponent (a number below |s| + log2 Sk, rounded twice), O is off by the same
share of sum_j P_j |v_j| of its column plus 12 Sk / 16 roundings of it (in the
worst case; the bar is not reached).
"""
import numpy as np
import pytest
import torch

from hipgpt_amd import attention as A

pytestmark = pytest.mark.gpu

# (B, H, S, D): small grids (key splits), middle, and larger than the device;
# padded head dims and lengths that are no multiple of a tile
SHAPES = [(1, 8, 256, 32), (2, 8, 300, 32), (16, 8, 200, 32), (64, 8, 130, 32), (1, 4, 256, 64), (2, 4, 333, 64),
          (20, 8, 257, 64), (70, 8, 100, 64), (2, 4, 200, 128), (20, 8, 190, 128), (70, 8, 129, 128), (2, 3, 70, 48),
          (3, 3, 90, 96), (40, 8, 150, 80), (3, 2, 61, 20), (7, 8, 180, 32), (4, 8, 290, 32), (7, 8, 180, 64),
          (6, 8, 600, 64), (12, 8, 170, 128)]


def make(B, H, S, D, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(3, B, S, H, D, generator=g)


def run(x, causal, probs):
    _, B, S, H, D = x.shape
    d = x.cuda().reshape(-1).contiguous()
    out = torch.full((B * S, H * D), 7.0, device="cuda")
    p = torch.full((B, H, S, S), 7.0, device="cuda") if probs else None
    A.qkv_planar(d, out, p, B, S, H * D, H, causal=causal)
    torch.cuda.synchronize()
    return out.cpu().reshape(B, S, H, D).double(), None if p is None else p.cpu().double()


def ref(x, causal):
    q, k, v = (t.permute(0, 2, 1, 3).double() for t in x)
    s = torch.matmul(q, k.transpose(-1, -2)) / np.sqrt(q.shape[-1])
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    return torch.matmul(p, v).permute(0, 2, 1, 3), p, s


def bars(x, p, s):
    """Bounds of |O - O64| and |P - P64| / P64, elementwise."""
    q, k, v = (t.permute(0, 2, 1, 3).double() for t in x)
    D, Sk = q.shape[-1], k.shape[-2]
    mag = torch.matmul(q.abs(), k.abs().transpose(-1, -2)) * (1.4427 * D ** -0.5)
    smax = torch.where(p > 0, s.abs() * 1.4427, 0.0).amax(-1, keepdim=True)
    rel = (mag * (2 + 12 * D / 16) + s.abs().where(p > 0, 0.0) * 1.4427 + smax) * 2.0 ** -24 * 0.6932 + 2.0 ** -22
    row = torch.where(p > 2.0 ** -60, rel, 0.0).amax(-1, keepdim=True) + Sk / 2 * 2.0 ** -24  # of the row's sum
    o = torch.matmul(p * (rel + row + (2 + 12 * Sk / 16) * 2.0 ** -24), v.abs())
    return o.permute(0, 2, 1, 3), rel + row + 2 * (smax + np.log2(Sk)) * 2.0 ** -24 * 0.6932


SCALES = [(1, 1, 1), (1e-6, 1, 1), (1, 1e-6, 1), (1, 1, 1e-6), (1, 1, 2.0 ** -12), (300, 1e-3, 1), (1e-3, 900, 1),
          (1e-4, 1e4, 1), (1, 1, 200), (1, 1, 1e15), (1e-30, 1, 1e30), (1e-30, 1e30, 1e-30), (1, 1, 0)]


def check(x, causal, probs, tag):
    o, p = run(x, causal, probs)
    want, pw, s = ref(x, causal)
    bo, bp = bars(x, pw, s)
    floor = 2.0 ** -126 * x.shape[2]  # exponentials below fp32's smallest normal are 0
    err = (o - want).abs() - floor * x[2].double().abs().amax(1, keepdim=True)
    print(tag, tuple(x.shape[1:]), causal, probs, "%.3f of the bar" % float((err / bo.clamp_min(1e-300)).max()), flush=True)
    assert (err <= bo + 1e-44).all()
    if probs:
        assert ((p - pw).abs() <= pw * bp + 2.0 ** -126).all()


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("probs", [False, True])
def test_scales(shape, probs):
    B, H, S, D = shape
    for i, scale in enumerate(SCALES):
        if B > 8 and i not in (0, 3, 5, 6):
            continue
        x = make(*shape, seed=i) * torch.tensor(scale, dtype=torch.float32).view(3, 1, 1, 1, 1)
        check(x, i % 2 == 0, probs, scale)


@pytest.mark.parametrize("shape", [SHAPES[i] for i in (0, 1, 3, 5, 6, 7, 9, 12)], ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("probs", [False, True])
def test_mixed_scales(shape, probs):
    B, H, S, D = shape
    for r in (2.0 ** 14, 2.0 ** 22, 2.0 ** 40):
        x = make(*shape, seed=20)
        x[0, ..., 0] *= r  # a feature large in Q and small in K
        x[1, ..., 0] /= r
        check(x, True, probs, "feature times %g" % r)
    for r in (1e-5, 1e-10, 1e-30):
        x = make(*shape, seed=21)
        x[2, ..., 1] *= r  # a small column of V
        x[2, :, :, :, 3] *= 1 / r ** 0.5
        check(x, False, probs, "column of V times %g" % r)
        x = make(*shape, seed=22)
        x[2, :, :32] *= r  # causal: rows that see the small values only
        check(x, True, probs, "first rows of V times %g" % r)
    x = make(*shape, seed=23) * torch.tensor([1, 1, 1e-7], dtype=torch.float32).view(3, 1, 1, 1, 1)
    x[2, 0, S - 1, 0, 0] = 2e-3
    check(x, True, probs, "one larger value of V")


@pytest.mark.parametrize("shape", [SHAPES[i] for i in (0, 1, 5, 6, 9, 12)], ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("probs", [False, True])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 1e35, 7e4])
def test_outlier(shape, probs, value):
    """One extreme entry of V: the rows of its (batch, head) get it with their
    weight, in its column only; one of K or Q: the softmax of the reference
    arithmetic in float32 says where O stays finite.  (1e35: exponentials reach
    2^8 before the running max is raised, and 2^8 * 64 keys of them still fit.)"""
    B, H, S, D = shape
    b, s, h, d = B - 1, S // 2, H - 1, D - 1
    for which in (2, 1, 0):
        x = make(*shape, seed=which)
        x[which, b, s, h, d] = value
        if which < 2 and np.isfinite(value) and value > 1e30:
            continue  # products overflow or not by the order of the sum
        o, _ = run(x, False, probs)
        want, _, sc = ref(x, False)
        # every other (batch, head), and for V every other column, as without it
        clean, _, _ = ref(make(*shape, seed=which), False)
        keep = torch.ones_like(o, dtype=torch.bool)
        if which == 2:
            keep[b, :, h, d] = False
        elif which == 1:
            keep[b, :, h, :] = False
        else:
            keep[b, s, h, :] = False
        assert torch.isfinite(o[keep]).all()
        assert float((o[keep] - clean[keep]).abs().max()) <= 1e-5
        bad = ~keep
        if which == 2 and np.isfinite(value):
            assert ((o[bad] - want[bad]).abs() <= 1e-5 * value).all()
        elif which == 2:
            assert torch.isnan(o[bad]).all() if np.isnan(value) else (o[bad] == value).all()
        elif np.isnan(value):
            assert torch.isnan(o[bad]).all()
        elif np.isfinite(value):
            rel = D * 2.0 ** -24 * float(sc.abs().max()) * 1.4427
            assert float((o[bad] - want[bad]).abs().max()) <= float(x[2].abs().max()) * (rel + 1e-6)


@pytest.mark.parametrize("shape", [SHAPES[i] for i in (0, 1, 4, 5, 6, 7, 9, 11)], ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("causal", [False, True])
def test_output_over_q(shape, causal):
    """O in Q's place, also where a workgroup takes the second pass: it starts
    from Q again, so nothing may be stored before."""
    B, H, S, D = shape
    for scale in ((1, 1, 1), (300, 1e-2, 1), (1, 1, 1e-6), (1, 1, 1e33)):
        x = (make(*shape, seed=5) * torch.tensor(scale, dtype=torch.float32).view(3, 1, 1, 1, 1)).cuda()
        q, k, v = x.unbind(0)
        want = A.attention(q, k, v, causal=causal)
        got = A.attention(q, k, v, out=q, causal=causal)
        assert got.data_ptr() == x.data_ptr()
        assert torch.equal(got, want), scale
