"""GPU tests of the split-operand forward (hipgpt_amd/csrc/split.h) at the
edges of its range: fp32 operands run as two fp16 terms, with scales that hold
for ordinary data, and a workgroup whose data lie outside runs again on fp32
MFMA.  Here Q, K and V come at scales on both sides of every limit, with
single outliers, and with infinities and NaN, in each workgroup shape of the
dispatch and at ragged sizes.

Finite cases against float64.  A score is a D-term fp32 sum of magnitude at
most smax (log2 units), so its error is below about D * 2^-24 * smax and that
of P the same, relatively; O is a P-weighted mean of V, so its error is at most
vmax times that plus the rounding of the products and of the sums over keys
(tiles of 32 in sequence): bar = vmax * (2^-22 + D 2^-24 smax + Sk / 32 * 2^-24).
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
          (3, 3, 90, 96), (40, 8, 150, 80), (3, 2, 61, 20)]


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


SCALES = [(1, 1, 1), (1e-6, 1, 1), (1, 1e-6, 1), (1, 1, 1e-6), (1, 1, 2.0 ** -9), (1, 1, 2.0 ** -12), (300, 1e-3, 1),
          (1e-3, 900, 1), (1e-4, 1e4, 1), (1, 1, 200), (1, 1, 1e4), (1e-30, 1, 1e30), (1, 1, 0)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%dH%dS%dD%d" % s)
@pytest.mark.parametrize("probs", [False, True])
def test_scales(shape, probs):
    B, H, S, D = shape
    for i, (sq, sk, sv) in enumerate(SCALES):
        if B > 8 and i not in (0, 3, 6, 7):
            continue
        x = make(*shape, seed=i) * torch.tensor([sq, sk, sv], dtype=torch.float32).view(3, 1, 1, 1, 1)
        causal = i % 2 == 0
        o, p = run(x, causal, probs)
        want, pw, s = ref(x, causal)
        smax = float(s[s > -1e300].abs().max()) * 1.4427
        rel = 2.0 ** -22 + D * 2.0 ** -24 * smax + S / 32 * 2.0 ** -24
        vmax = float(x[2].abs().max())
        err = float((o - want).abs().max())
        print(shape, probs, (sq, sk, sv), err, vmax * rel, flush=True)
        assert err <= vmax * rel
        if probs:
            assert float((p - pw).abs().max()) <= rel


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
