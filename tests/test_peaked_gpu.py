"""Parity on peaked logits: Q scaled by 8 and by 64 (scores with a standard
deviation of 8 and 64 instead of 1, as a trained layer's are), and the
argmax limit (Q scaled by 1e4).

These inputs make the online softmax move its running max far and often
(the lazy rescale, which only rescales O once a row max grows by more than
2^8), and they run the score-resident, recomputed and spilled probs sweeps
with scores far from the unit-variance range.

Shapes: c1 (D=32, streaming kernel, scores kept in registers with probs),
c2 (D=64, S=256, B*H=256), c3 (D=64, S=1024: Q.K^T recomputed with probs) and c4's head shape at B=1
(D=128, S=2048: probs rows spilled and read back).

Bars.  fp32 rounding of a score s costs about eps*|s|, and |s| grows with the
scale, so the unit-variance bars (1e-4 on O, 1e-5 on P) cannot hold for any
fp32 arithmetic at scale 64 (the oracle's own restatement of the reference
kernels is 1.8e-4 from the float64 closed form on O at c3, 4.4e-5 on P).
So each comparison is held to
* O: max|dO| <= 1e-4 * max(1, max|O|) against the reference's launcher
  (non-causal) or the oracle (causal), and the HIP error against float64 at
  most 3x the reference arithmetic's error against float64, plus 1e-5;
* P: max|dP| <= max(1e-5, 3 * the reference arithmetic's own max|dP|
  against float64), against the reference / oracle and against float64.
The reference arithmetic is src/hip_kernels.cpp:263-325 (flash) and
:329-402 (fallback), run as the reference's own launcher (oracle/_ref) for
the non-causal drop-in call and as the oracle restatement for causal.
"""
import numpy as np
import pytest
import torch

import oracle as O
from hipgpt_amd import attention as A

pytestmark = pytest.mark.gpu

SEED = 0x48495047
NT = 16

SHAPES = {  # name: (B, H, S, D, seed index)
    "c1": (32, 8, 256, 32, 0),
    "c2": (32, 8, 256, 64, 1),
    "c3": (8, 12, 1024, 64, 2),
    "c4_b1": (1, 16, 2048, 128, 3),
}


def dev_t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda")


def host(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def scaled_planar(name, scale):
    B, H, S, D, idx = SHAPES[name]
    E = H * D
    qkv = O.seeded_planar(SEED + idx, B, S, E).copy()
    qkv[: B * S * E] *= np.float32(scale)
    return qkv, B, H, S, D, E


def f64_planar(qkv, B, S, E, H, causal):
    q, k, v = O.planar_qkv(qkv, B, S, E, H)
    o, p = O.attention(q, k, v, causal=causal, f64=True, want_probs=True, nthreads=NT)
    return o.reshape(B * S, E), p


def run_hip(d_qkv, B, S, E, H, causal, with_probs):
    out = torch.full((B * S, E), float("nan"), device="cuda")
    p = torch.full((B, H, S, S), float("nan"), device="cuda") if with_probs else None
    if causal:
        A.qkv_planar(d_qkv, out, p, B, S, E, H, causal=True)
    else:
        A.launch_multihead_attention(d_qkv, out, p, B, S, E, H)
    return host(out), (host(p) if with_probs else None)


def mx(a, b):
    return float(np.abs(a.astype(np.float64) - b).max())


def check(name, got_o, got_p, cmp_o, cmp_p, o64, p64):
    """HIP output against the reference arithmetic (cmp) and float64."""
    assert np.isfinite(got_o).all()
    bar_o = 1e-4 * max(1.0, float(np.abs(o64).max()))
    e_ref_o = mx(cmp_o, o64)
    e_hip_o = mx(got_o, o64)
    d_o = mx(got_o, cmp_o)
    line = f"[{name}] |dO| vs ref {d_o:.2e} (bar {bar_o:.2e}); vs f64 hip {e_hip_o:.2e} ref {e_ref_o:.2e}"
    if got_p is not None:
        assert np.isfinite(got_p).all()
        e_ref_p = mx(cmp_p, p64)
        bar_p = max(1e-5, 3 * e_ref_p)
        e_hip_p = mx(got_p, p64)
        d_p = mx(got_p, cmp_p)
        line += f"; |dP| vs ref {d_p:.2e} vs f64 hip {e_hip_p:.2e} ref {e_ref_p:.2e} (bar {bar_p:.2e})"
    print(line, flush=True)
    assert d_o <= bar_o
    assert e_hip_o <= 3 * e_ref_o + 1e-5
    if got_p is not None:
        assert d_p <= bar_p
        assert e_hip_p <= bar_p


@pytest.mark.parametrize("scale", [8, 64])
@pytest.mark.parametrize("name", list(SHAPES))
def test_peaked_dropin_matches_reference_launcher(dev, name, scale):
    """HipGPT's call (non-causal, probs written, and without probs) on
    peaked logits against the reference's own launcher on the same buffers."""
    if not O.ref_available():
        pytest.skip("reference build oracle/_ref missing")
    ref = O.ref_lib()
    qkv, B, H, S, D, E = scaled_planar(name, scale)
    print(f"\n[{name} x{scale}] drop-in B={B} H={H} S={S} D={D}", flush=True)
    d_qkv = dev_t(qkv)
    r_out = torch.zeros((B * S, E), device=dev)
    r_p = torch.zeros((B, H, S, S), device=dev)
    ref.launch(d_qkv.data_ptr(), r_out.data_ptr(), r_p.data_ptr(), B, S, E, H)
    cmp_o, cmp_p = host(r_out), host(r_p)
    del r_out, r_p
    o64, p64 = f64_planar(qkv, B, S, E, H, causal=False)
    got_o, got_p = run_hip(d_qkv, B, S, E, H, causal=False, with_probs=True)
    check(f"{name} x{scale} probs", got_o, got_p, cmp_o, cmp_p, o64, p64)
    del got_p
    got_o2, _ = run_hip(d_qkv, B, S, E, H, causal=False, with_probs=False)
    check(f"{name} x{scale} no probs", got_o2, None, cmp_o, None, o64, None)


@pytest.mark.parametrize("scale", [8, 64])
@pytest.mark.parametrize("name", list(SHAPES))
def test_peaked_causal_matches_oracle(dev, name, scale):
    """Causal, with and without probs, on peaked logits against the oracle's
    restatement (keys j <= i) and float64."""
    qkv, B, H, S, D, E = scaled_planar(name, scale)
    print(f"\n[{name} x{scale}] causal B={B} H={H} S={S} D={D}", flush=True)
    cmp_o, cmp_p = O.launch_multihead_attention(qkv, B, S, E, H, causal=True, want_probs=True, nthreads=NT)
    o64, p64 = f64_planar(qkv, B, S, E, H, causal=True)
    d_qkv = dev_t(qkv)
    got_o, got_p = run_hip(d_qkv, B, S, E, H, causal=True, with_probs=True)
    check(f"{name} x{scale} causal probs", got_o, got_p, cmp_o, cmp_p, o64, p64)
    assert np.all(np.triu(got_p, 1) == 0.0)
    del got_p
    got_o2, _ = run_hip(d_qkv, B, S, E, H, causal=True, with_probs=False)
    check(f"{name} x{scale} causal", got_o2, None, cmp_o, None, o64, None)
    if D in (32, 64):
        out = torch.full((B * S, E), float("nan"), device=dev)
        lse = torch.full((B * H * S,), float("nan"), device=dev)
        A.fwd_lse_qkv_planar(d_qkv, out, lse, B, S, E, H, causal=True)
        check(f"{name} x{scale} causal lse", host(out), None, cmp_o, None, o64, None)
        assert np.isfinite(host(lse)).all()


def _argmax_rows(qkv, B, S, E, H, causal):
    """Per (b, h, i): the index of the largest score (float64), and whether
    it beats the runner-up by more than 50 (natural-log units of the scaled
    score), so that every other probability is below e^-50."""
    D = E // H
    q, k, _ = O.planar_qkv(qkv, B, S, E, H)
    qt = np.ascontiguousarray(q.transpose(0, 2, 1, 3), dtype=np.float64)
    kt = np.ascontiguousarray(k.transpose(0, 2, 3, 1), dtype=np.float64)
    s = np.matmul(qt, kt) / np.sqrt(D)  # [B, H, S, S]
    if causal:
        s[..., np.triu_indices(S, 1)[0], np.triu_indices(S, 1)[1]] = -np.inf
    top2 = np.partition(s, S - 2, axis=-1)[..., S - 2:] if S > 1 else None
    am = s.argmax(-1)
    if S > 1:
        gap = top2[..., 1] - top2[..., 0]
        clean = gap > 50.0
        if causal:
            clean[..., 0] = True  # row 0 sees one key
    else:
        clean = np.ones(am.shape, dtype=bool)
    return am, clean


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("name", ["c1", "c3"])
def test_argmax_limit(dev, name, causal):
    """Q scaled by 1e4: every output finite; where the top score beats the
    runner-up by more than 50, O is V of the argmax key and P that row's
    one-hot vector (within 1e-5)."""
    qkv, B, H, S, D, E = scaled_planar(name, 1e4)
    print(f"\n[{name} x1e4] argmax causal={causal}", flush=True)
    am, clean = _argmax_rows(qkv, B, S, E, H, causal)
    assert clean.mean() > 0.9
    _, _, v = O.planar_qkv(qkv, B, S, E, H)
    want = np.take_along_axis(v.transpose(0, 2, 1, 3), am[..., None], axis=2)  # [B, H, S, D]
    d_qkv = dev_t(qkv)
    got_o, got_p = run_hip(d_qkv, B, S, E, H, causal=causal, with_probs=True)
    assert np.isfinite(got_o).all() and np.isfinite(got_p).all()
    go = got_o.reshape(B, S, H, D).transpose(0, 2, 1, 3)
    err_o = float(np.abs(go - want)[clean].max())
    onehot_err = float(np.abs(np.take_along_axis(got_p, am[..., None], axis=-1)[..., 0] - 1.0)[clean].max())
    rest = got_p.copy()
    np.put_along_axis(rest, am[..., None], 0.0, axis=-1)
    rest_err = float(np.abs(rest).max(-1)[clean].max())
    print(f"[{name} x1e4] clean rows {clean.mean():.3f}: |O - V[argmax]| {err_o:.2e}, "
          f"|P[argmax] - 1| {onehot_err:.2e}, max other P {rest_err:.2e}", flush=True)
    assert err_o <= 1e-5 and onehot_err <= 1e-5 and rest_err <= 1e-5
    got_o2, _ = run_hip(d_qkv, B, S, E, H, causal=causal, with_probs=False)
    assert np.isfinite(got_o2).all()
    go2 = got_o2.reshape(B, S, H, D).transpose(0, 2, 1, 3)
    assert float(np.abs(go2 - want)[clean].max()) <= 1e-5
