#!/usr/bin/env python3
"""Benchmark of the MI355X attention forward (HipGPT's hot path) on one GPU.

Headline: causal attention forward TFLOP/s and the fraction of the roofline of
fp32 products on the matrix cores at B32 H8 S256 D32 (config c1), inputs
resident in HBM.  One step = one attention forward over the whole batch.
The other configs, the drop-in contract (non-causal + probs, the call HipGPT
makes) at every config, and the neighbouring kernels are timed the same way; the
oracle's scalar restatement is timed on the host cores for c1..c5.

stdout is one JSON line of under 4 KB: the headline, and per config under
"configs" its microseconds per call and roofline fraction.  stderr has a readable
line per config; --details FILE takes everything measured, as JSON.

Timing protocol, per config:
  * Input and output buffers are allocated in R independent sets, R chosen so
    the sets together hold at least 1 GiB; timed calls rotate over the sets,
    so a set is evicted from the 256 MB Infinity Cache (and every L2) before
    it is used again and each call reads its operands from HBM.  This is
    "us_per_call", the figure every rate and roofline fraction is computed
    from.  "us_per_call_hot" repeats the calls on one set (operands can stay
    in the Infinity Cache between calls).
  * Both are means over exactly --steps back-to-back calls between two HIP
    events on the launch stream, after >= 0.2 s of untimed calls (the GPU
    needs ~0.1 s of load to reach its steady clock).
  * "dist_us": p10 / p50 / p90 over max(steps, 100) calls, each between its
    own pair of events (rotating sets).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--only c1,c3] [--no-cpu] [--no-hot] [--details FILE]
"""
import argparse
import json
import math
import os
import platform
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_BF16_MFMA = 2.5e15    # MI355X dense bf16 matrix, FLOP/s
# fp32 products at fp32 accuracy: six bf16 MFMAs each (hipgpt_amd/csrc/terms.h),
# 2.6 times the dense fp32 matrix rate
PEAK_F32_MFMA = PEAK_BF16_MFMA / 6
RATE_F32_MFMA = 157.3e12   # dense fp32 matrix
PEAK_HBM = 8.0e12          # HBM3E bytes/s
METRIC = "causal attention fwd TFLOP/s + % of MFMA roofline on 1 MI355X (B32 H8 S256 D32)"
ROTATE_BYTES = 1 << 30     # buffer sets per config hold at least this much together
SEED = 0x48495047

# name: (B, H, Sq, Sk, D, causal, dtype, probs, kind)
# "legacy" lines are the drop-in call HipGPT makes (src/transformer_layer.cpp:
# 208, 218-219): non-causal, probs written, through launch_multihead_attention
# on the null stream.  "probs" lines are causal with probs (extended API).
CONFIGS = {
    "c1": (32, 8, 256, 256, 32, True, "f32", False, "fwd"),
    "c1_probs": (32, 8, 256, 256, 32, True, "f32", True, "fwd"),
    "c1_legacy": (32, 8, 256, 256, 32, False, "f32", True, "fwd"),
    "c2": (32, 8, 256, 256, 64, True, "f32", False, "fwd"),
    "c2_probs": (32, 8, 256, 256, 64, True, "f32", True, "fwd"),
    "c2_legacy": (32, 8, 256, 256, 64, False, "f32", True, "fwd"),
    "c3": (8, 12, 1024, 1024, 64, True, "f32", False, "fwd"),
    "c3_probs": (8, 12, 1024, 1024, 64, True, "f32", True, "fwd"),
    "c3_legacy": (8, 12, 1024, 1024, 64, False, "f32", True, "fwd"),
    "c3_bf16": (8, 12, 1024, 1024, 64, True, "bf16", False, "fwd"),
    "c4": (4, 16, 2048, 2048, 128, True, "f32", False, "fwd"),
    "c4_probs": (4, 16, 2048, 2048, 128, True, "f32", True, "fwd"),
    "c4_legacy": (4, 16, 2048, 2048, 128, False, "f32", True, "fwd"),
    "c5": (64, 12, 1, 2048, 64, False, "f32", False, "decode"),
    # c5 as a KV-cache step: 2047 cached rows + the new one appended in place
    "c5_kvcache": (64, 12, 1, 2048, 64, False, "f32", False, "kvcache"),
    # One long sequence: few (b, h) rows, so the keys are split over 64
    # workgroups per row and the reduce kernel merges them.
    "decode_long": (1, 12, 1, 32768, 64, False, "f32", False, "decode"),
    # The c1 head shape at other batch sizes: HipGPT's generation call
    # (GPTModel::generate, src/gpt_model.cpp:273: B = 1, non-causal, probs)
    # and a batch whose grid is four times the device's resident slots.
    "gen_b1_legacy": (1, 8, 256, 256, 32, False, "f32", True, "fwd"),
    "c1_b128": (128, 8, 256, 256, 32, True, "f32", False, "fwd"),
    "c1_b128_legacy": (128, 8, 256, 256, 32, False, "f32", True, "fwd"),
    # HipGPT's unfused single-head helpers (include/hip_kernels.h:44-46) at the
    # c1 shape with batch and heads merged (B*H = 256 sequences of 256 x 32).
    "a8_scores": (256, 1, 256, 256, 32, False, "f32", False, "sdp"),
    "a8_softmax": (256, 1, 256, 256, 32, False, "f32", False, "softmax"),
    "a8_wsum": (256, 1, 256, 256, 32, False, "f32", False, "wsum"),
    # Attention backward on the forward's probs (src/hip_kernels.cpp:1159-1272)
    # at the c1 / c2 shapes: causal through the extended entry point, and the
    # drop-in symbol on non-causal probs.
    "c1_bwd": (32, 8, 256, 256, 32, True, "f32", True, "bwd"),
    "c1_bwd_legacy": (32, 8, 256, 256, 32, False, "f32", True, "bwd"),
    "c2_bwd": (32, 8, 256, 256, 64, True, "f32", True, "bwd"),
    "c2_bwd_legacy": (32, 8, 256, 256, 64, False, "f32", True, "bwd"),
    # ... and at the c3 / c4 shapes (D = 64 and 128, long rows).
    "c3_bwd": (8, 12, 1024, 1024, 64, True, "f32", True, "bwd"),
    "c3_bwd_legacy": (8, 12, 1024, 1024, 64, False, "f32", True, "bwd"),
    "c4_bwd": (4, 16, 2048, 2048, 128, True, "f32", True, "bwd"),
    "c4_bwd_legacy": (4, 16, 2048, 2048, 128, False, "f32", True, "bwd"),
    # A head dim above 128 (the reference fallback takes any D = E / H):
    # forward causal and as the drop-in, and the drop-in backward.
    "d256": (4, 8, 1024, 1024, 256, True, "f32", False, "fwd"),
    "d256_legacy": (4, 8, 1024, 1024, 256, False, "f32", True, "fwd"),
    "d256_bwd_legacy": (4, 8, 1024, 1024, 256, False, "f32", True, "bwd"),
    "d512": (2, 4, 1024, 1024, 512, True, "f32", False, "fwd"),
    # The probs-free training pair at the same shapes: forward writing O and the
    # row log-sum-exp, and the backward that recomputes P from it.
    "c1_fwd_lse": (32, 8, 256, 256, 32, True, "f32", False, "fwd_lse"),
    "c1_bwd_lse": (32, 8, 256, 256, 32, True, "f32", False, "bwd_lse"),
    "c2_bwd_lse": (32, 8, 256, 256, 64, True, "f32", False, "bwd_lse"),
    "c4_fwd_lse": (4, 16, 2048, 2048, 128, True, "f32", False, "fwd_lse"),
    "c4_bwd_lse": (4, 16, 2048, 2048, 128, True, "f32", False, "bwd_lse"),
    # The projections either side of the attention (launch_matmul_add_bias,
    # src/transformer_layer.cpp:217, :220) as (M, N, K, -, -, ...): the c1
    # layer (T = 8192 tokens, E = 256) and the GPT-2-small c3 layer (E = 768).
    "gemm_qkv_c1": (8192, 768, 256, 0, 0, False, "f32", False, "gemm"),
    "gemm_out_c1": (8192, 256, 256, 0, 0, False, "f32", False, "gemm"),
    "gemm_qkv_c3": (8192, 2304, 768, 0, 0, False, "f32", False, "gemm"),
    "gemm_out_c3": (8192, 768, 768, 0, 0, False, "f32", False, "gemm"),
    # HipGPT's attention block as TransformerLayer::self_attention_forward
    # issues it (src/transformer_layer.cpp:214-222): QKV projection into the
    # [T][3E] buffer, the drop-in attention on it (non-causal, probs written),
    # output projection -- three launches on the null stream per call.
    "c1_layer": (32, 8, 256, 256, 32, False, "f32", True, "layer"),
}


def work(cfg):
    """Algorithmic FLOPs (4*B*H*D*P, P visible pairs) and HBM bytes (Q, K, V
    read once, O written once, plus probs when written)."""
    B, H, Sq, Sk, D, causal, dtype, probs, kind = cfg
    if kind == "gemm":  # A [M, K] @ W [K, N] + bias: read A, W, bias; write C
        M, N, K = B, H, Sq
        return 2.0 * M * N * K, 4 * (M * K + K * N + N + M * N)
    if kind == "layer":  # the three calls' work, each counted as its own line counts it
        T, E = B * Sq, H * D
        parts = [work((T, 3 * E, E, 0, 0, False, "f32", False, "gemm")),
                 work((B, H, Sq, Sk, D, causal, dtype, probs, "fwd")),
                 work((T, E, E, 0, 0, False, "f32", False, "gemm"))]
        return sum(f for f, _ in parts), sum(b for _, b in parts)
    if kind == "sdp":  # read Q, K; write scores
        return 2.0 * B * Sq * Sk * D, 4 * (2 * B * Sq * D + B * Sq * Sk)
    if kind == "softmax":  # read and write B*S*S (no flops counted)
        return 0.0, 8 * B * Sq * Sk
    if kind == "wsum":  # read P, V; write O
        return 2.0 * B * Sq * Sk * D, 4 * (B * Sq * Sk + 2 * B * Sq * D)
    if kind == "bwd":
        # dP, dV, dQ, dK: 8 D flops per visible pair; read the visible probs,
        # Q, K, V, dO; write dQ, dK, dV
        pairs = Sq * (Sq + 1) // 2 if causal else Sq * Sk
        return 8.0 * B * H * D * pairs, 4 * B * H * (pairs + 7 * Sq * D)
    if kind == "bwd_lse":
        # dP, dV, dQ, dK: 8 D flops per visible pair; read Q, K, V, O, dO and
        # the lse; write dQ, dK, dV
        pairs = Sq * (Sq + 1) // 2 if causal else Sq * Sk
        return 8.0 * B * H * D * pairs, 4 * B * H * (8 * Sq * D + Sq)
    if kind == "fwd_lse":  # the forward's bytes plus the lse row
        pairs = Sq * (Sq + 1) // 2 if causal else Sq * Sk
        return 4.0 * B * H * D * pairs, 4 * B * H * (4 * Sq * D + Sq)
    if kind == "kvcache":
        # read the 2047 cached rows and the new row, q; write the new row into
        # the cache and O
        return 4.0 * B * H * D * Sk, 4 * B * H * D * (2 * (Sk - 1) + 2 + 1 + 2 + 1)
    if kind == "decode":
        pairs = Sk
    elif causal:
        off = Sk - Sq
        pairs = sum(min(Sk, i + 1 + off) for i in range(Sq))
    else:
        pairs = Sq * Sk
    flops = 4.0 * B * H * D * pairs
    el = 2 if dtype == "bf16" else 4
    nbytes = el * B * H * D * (Sq + 2 * Sk) + 4 * B * H * Sq * D
    if probs:
        nbytes += 4 * B * H * Sq * Sk
    return flops, nbytes


def set_bytes(cfg):
    """Device bytes of one input + output set of a config (for the rotation count)."""
    B, H, Sq, Sk, D, causal, dtype, probs, kind = cfg
    if kind == "gemm":
        M, N, K = B, H, Sq
        return 4 * (M * K + K * N + N + M * N)
    if kind == "layer":  # x, W_qkv, b_qkv, qkv, attention out, probs, W_out, b_out, y
        T, E = B * Sq, H * D
        return 4 * (T * E + E * 3 * E + 3 * E + 3 * T * E + T * E + B * H * Sq * Sk + E * E + E + T * E)
    if kind in ("sdp", "softmax", "wsum"):
        return 4 * (3 * B * Sq * D + 2 * B * Sq * Sk + B * Sq * D)
    E = H * D
    if kind == "bwd":
        return 4 * (3 * B * Sq * E + B * Sq * E + B * Sq * E + B * H * Sq * Sk + 3 * B * Sq * E)
    if kind in ("fwd_lse", "bwd_lse"):
        return 4 * (3 * B * Sq * E + 2 * B * Sq * E + B * H * Sq + 3 * B * Sq * E)
    if kind in ("decode", "kvcache"):
        return 4 * B * H * D * (2 * Sk + 4)
    el = 2 if dtype == "bf16" else 4
    return el * B * H * D * (Sq + 2 * Sk) + 4 * B * H * Sq * D + (4 * B * H * Sq * Sk if probs else 0)


def make_call(cfg, torch, A, dev, seed=SEED):
    """One input/output set of a config and the call that runs it.
    Returns (fn, extra)."""
    B, H, Sq, Sk, D, causal, dtype, probs, kind = cfg
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    if kind == "decode":
        q = torch.randn(B, 1, H, D, device=dev, generator=g)
        k = torch.randn(B, Sk, H, D, device=dev, generator=g)
        v = torch.randn(B, Sk, H, D, device=dev, generator=g)
        out = torch.empty(B, 1, H, D, device=dev)
        ns = A.decode_default_splits(B, H, Sk)
        ws = torch.empty(max(1, A.decode_workspace_bytes(B, H, D, ns) // 4), device=dev)
        return (lambda: A.decode(q, k, v, out=out, num_splits=ns, workspace=ws),
                {"splits": ns, "entry": "hipgpt_attn_decode"})
    if kind == "kvcache":
        kc = torch.randn(B, Sk, H, D, device=dev, generator=g)
        vc = torch.randn(B, Sk, H, D, device=dev, generator=g)
        q, kn, vn = torch.randn(3, B, H, D, device=dev, generator=g)
        out = torch.empty(B, H, D, device=dev)
        lens = torch.full((B,), Sk - 1, dtype=torch.int32, device=dev)
        ns = A.decode_default_splits(B, H, Sk)
        ws = torch.empty(max(1, A.decode_workspace_bytes(B, H, D, ns) // 4), device=dev)
        # advance=False: every timed call is the same step (row Sk-1 rewritten)
        return (lambda: A.decode_kvcache(q, kn, vn, kc, vc, lens, out=out, advance=False, num_splits=ns,
                                         workspace=ws), {"splits": ns, "entry": "hipgpt_attn_decode_kvcache"})
    if kind == "gemm":
        from hipgpt_amd import projection as P

        M, N, K = B, H, Sq
        a = torch.randn(M, K, device=dev, generator=g)
        w = torch.randn(K, N, device=dev, generator=g)
        bias = torch.randn(N, device=dev, generator=g)
        c = torch.empty(M, N, device=dev)
        return (lambda: P.launch_matmul_add_bias(a, w, bias, c, M, K, N),
                {"entry": "launch_matmul_add_bias (null stream)", "M": M, "N": N, "K": K})
    if kind == "layer":
        from hipgpt_amd import projection as P

        T, E = B * Sq, H * D
        x = torch.randn(T, E, device=dev, generator=g)
        wqkv = torch.randn(E, 3 * E, device=dev, generator=g) * E ** -0.5
        bqkv = torch.randn(3 * E, device=dev, generator=g)
        wo = torch.randn(E, E, device=dev, generator=g) * E ** -0.5
        bo = torch.randn(E, device=dev, generator=g)
        qkv = torch.empty(T, 3 * E, device=dev)
        att = torch.empty(T, E, device=dev)
        p = torch.empty(B, H, Sq, Sk, device=dev)
        y = torch.empty(T, E, device=dev)

        def layer():
            P.launch_matmul_add_bias(x, wqkv, bqkv, qkv, T, E, 3 * E)
            A.launch_multihead_attention(qkv.view(-1), att, p, B, Sq, E, H)
            P.launch_matmul_add_bias(att, wo, bo, y, T, E, E)

        return layer, {"layer": "[T][3E] QKV buffer, as the reference layer passes it",
                       "entry": "launch_matmul_add_bias + launch_multihead_attention + launch_matmul_add_bias"}
    if kind in ("sdp", "softmax", "wsum"):
        x = torch.randn(3, B * Sq, D, device=dev, generator=g)
        sc = torch.randn(B * Sq, Sk, device=dev, generator=g)
        out = torch.empty(B * Sq, Sk, device=dev)
        o = torch.empty(B * Sq, D, device=dev)
        if kind == "sdp":
            return lambda: A.launch_scaled_dot_product(x[0], x[1], out, B, Sq, D), {"layout": "[B*S][D]"}
        if kind == "softmax":
            return lambda: A.launch_softmax(sc, out, B, Sq), {"layout": "[B*S][S]"}
        p = torch.softmax(sc, dim=-1).contiguous()
        return lambda: A.launch_attention_weighted_sum(p, x[2], o, B, Sq, D), {"layout": "[B*S][S] x [B*S][D]"}
    E = H * D
    if kind == "bwd":
        qkv = torch.randn(3 * B * Sq * E, device=dev, generator=g)
        go = torch.randn(B * Sq * E, device=dev, generator=g)
        out = torch.empty(B * Sq, E, device=dev)
        p = torch.empty(B, H, Sq, Sk, device=dev)
        A.qkv_planar(qkv, out, p, B, Sq, E, H, causal=causal)  # the probs the forward hands over
        grad = torch.empty(3 * B * Sq * E, device=dev)
        if not causal:
            return (lambda: A.launch_multihead_attention_backward(go, qkv, p, grad, B, Sq, E, H),
                    {"layout": "planar [3][B*S][E]", "entry": "launch_multihead_attention_backward"})
        ws = torch.empty(B * H * Sq, device=dev)
        return (lambda: A.attention_backward(go, qkv, p, grad, B, Sq, E, H, causal=True, workspace=ws),
                {"layout": "planar [3][B*S][E]", "entry": "hipgpt_attn_bwd_qkv_planar"})
    if kind in ("fwd_lse", "bwd_lse"):
        qkv = torch.randn(3 * B * Sq * E, device=dev, generator=g)
        out = torch.empty(B * Sq, E, device=dev)
        lse = torch.empty(B * H * Sq, device=dev)
        A.fwd_lse_qkv_planar(qkv, out, lse, B, Sq, E, H, causal=causal)
        if kind == "fwd_lse":
            return (lambda: A.fwd_lse_qkv_planar(qkv, out, lse, B, Sq, E, H, causal=causal),
                    {"layout": "planar [3][B*S][E]", "entry": "hipgpt_attn_fwd_lse_qkv_planar"})
        go = torch.randn(B * Sq * E, device=dev, generator=g)
        grad = torch.empty(3 * B * Sq * E, device=dev)
        ws = None if D in (32, 64) else torch.empty(B * H * Sq, device=dev)  # row dots dO . O
        return (lambda: A.bwd_lse_qkv_planar(go, qkv, out, lse, grad, B, Sq, E, H, causal=causal, workspace=ws),
                {"layout": "planar [3][B*S][E]", "entry": "hipgpt_attn_bwd_lse_qkv_planar"})
    if dtype == "f32" and Sq == Sk:
        # the reference's planar [Q|K|V] buffer
        qkv = torch.randn(3 * B * Sq * E, device=dev, generator=g)
        out = torch.empty(B * Sq, E, device=dev)
        p = torch.empty(B, H, Sq, Sk, device=dev) if probs else None
        if probs and not causal:  # the drop-in symbol, exactly as HipGPT calls it
            return (lambda: A.launch_multihead_attention(qkv, out, p, B, Sq, E, H),
                    {"layout": "planar [3][B*S][E]", "entry": "launch_multihead_attention (null stream)"})
        return (lambda: A.qkv_planar(qkv, out, p, B, Sq, E, H, causal=causal),
                {"layout": "planar [3][B*S][E]", "entry": "hipgpt_attn_qkv_planar"})
    q = torch.randn(B, Sq, H, D, device=dev, generator=g).to(tdt)
    k = torch.randn(B, Sk, H, D, device=dev, generator=g).to(tdt)
    v = torch.randn(B, Sk, H, D, device=dev, generator=g).to(tdt)
    out = torch.empty(B, Sq, H, D, device=dev)
    p = torch.empty(B, H, Sq, Sk, device=dev) if probs else None
    return (lambda: A.attention(q, k, v, out=out, probs=p, causal=causal),
            {"layout": "[B,S,H,D]", "entry": "hipgpt_attn_fwd"})


def warm_up(fns, warmup, torch, min_warm_s=0.2):
    """`warmup` calls and at least `min_warm_s` seconds of calls, rotating over
    the sets: the MI355X needs ~0.1 s of load to reach its steady clock, and
    an idle gap right before the timed calls would be timed at a lower clock."""
    n = 0
    t_end = time.perf_counter() + min_warm_s
    while n < warmup or time.perf_counter() < t_end:
        fns[n % len(fns)]()
        n += 1
        if n % 50 == 0:
            torch.cuda.synchronize()
    torch.cuda.synchronize()


def time_call(fns, steps, warmup, torch):
    """ms per call over exactly `steps` back-to-back calls (call i on set
    i % len(fns)), HIP events on the stream the calls launch on."""
    warm_up(fns, warmup, torch)
    stream = torch.cuda.current_stream()  # the stream the library launches on (the null stream here)
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for i in range(steps):
        fns[i % len(fns)]()
    stop.record(stream)
    torch.cuda.synchronize()
    return start.elapsed_time(stop) / steps


def launch_dist(fns, n, torch):
    """Per-call times (us) of n calls, each between its own pair of events;
    returns p10 / p50 / p90."""
    import numpy as np

    warm_up(fns, 0, torch)
    stream = torch.cuda.current_stream()
    ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]
    for i in range(n):
        ev[i][0].record(stream)
        fns[i % len(fns)]()
        ev[i][1].record(stream)
    torch.cuda.synchronize()
    t = np.array([a.elapsed_time(b) * 1e3 for a, b in ev])
    p10, p50, p90 = np.percentile(t, [10, 50, 90])
    return {"p10": round(float(p10), 3), "p50": round(float(p50), 3), "p90": round(float(p90), 3), "n": n}


# ------------------------------------------------------------ CPU baseline

CPU_CONFIGS = ("c1", "c2", "c3", "c4", "c5")


def host_info():
    model = platform.processor() or "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        affinity = len(os.sched_getaffinity(0))
    except AttributeError:
        affinity = os.cpu_count() or 1
    return {"cpu_model": model, "nproc": os.cpu_count(), "affinity": affinity}


def cpu_config(name, nthreads, budget_s):
    """The oracle's scalar restatement of the reference kernel HipGPT would run
    for config `name` (flash_attention_kernel passes for D in {32, 64} with
    S <= 512, the fallback's three-pass recompute otherwise; causal configs
    restricted to keys j <= i; c5 = the last row of the S = 2048 fallback,
    i.e. one query against 2048 keys) on the host cores.  Every (b, h) pair
    costs the same, so a subsample of evenly spaced pairs is timed and scaled
    by B*H / pairs: the pair count doubles from `nthreads` until one run takes
    at least budget_s / 3 (or covers every pair), then runs repeat until
    budget_s / 2 has elapsed; the median run is reported."""
    import statistics

    import oracle as O

    B, H, Sq, Sk, D, causal, dtype, probs, kind = CONFIGS[name]
    variant = O.FLASH if (kind == "fwd" and D in (32, 64) and Sk <= 512) else O.FALLBACK
    q, k, v = O.seeded_bshd(SEED, B, Sq, Sk, H, D)
    allp = [(b, h) for b in range(B) for h in range(H)]

    def pick(n):
        step = len(allp) / n
        return [allp[int(i * step)] for i in range(n)]

    def run(n):
        pr = pick(n)
        t0 = time.perf_counter()
        O.attention(q, k, v, causal=causal, variant=variant, nthreads=nthreads, pairs=pr)
        return time.perf_counter() - t0

    n = min(nthreads, len(allp))
    dt = run(n)
    while dt < budget_s / 3 and n < len(allp):
        n = min(2 * n, len(allp))
        dt = run(n)
    times = [dt]
    while sum(times) < budget_s / 2:
        times.append(run(n))
    dt = statistics.median(times)
    flops, _ = work(CONFIGS[name])
    us = dt * len(allp) / n * 1e6
    return {"us_per_call": round(us, 1), "gflops": round(flops / (us * 1e-6) / 1e9, 3), "threads": nthreads,
            "pairs": n, "of_pairs": len(allp), "runs": len(times),
            "variant": "flash" if variant == O.FLASH else "fallback"}


def cpu_baseline(budget_1t=3.0, budget_all=1.5):
    """c1..c5 at 1 thread and at all usable host cores (the box's CPU share
    for one GPU is 16 threads, whatever nproc reports)."""
    info = host_info()
    ncores = max(1, min(16, info["affinity"]))
    cfgs = {}
    for name in CPU_CONFIGS:
        one = cpu_config(name, 1, budget_1t)
        alln = cpu_config(name, ncores, budget_all)
        cfgs[name] = {"one_thread": one, "all_cores": alln}
        print(f"# cpu {name}: 1 thread {one['us_per_call']:.0f} us ({one['pairs']}/{one['of_pairs']} pairs), "
              f"{ncores} threads {alln['us_per_call']:.0f} us", file=sys.stderr, flush=True)
    return info, ncores, cfgs


def read_traffic(name):
    path = os.path.join(ROOT, "profiles", f"traffic_{name}.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f).get("hbm_bytes_per_launch")


def headline(steps, warmup, results, cpu):
    """The JSON line: c1 and, in short, every config of `results`."""
    head = results.get("c1", {})
    line = {
        "metric": METRIC,
        "value": head.get("tflops"),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": round(head["us_per_call"] / 1e3, 6) if "us_per_call" in head else None,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic N(0,1) Q/K/V resident in HBM (planar [3][B*S][E] buffer, seeded; calls rotate "
                "over buffer sets totalling >= 1 GiB so operands come from HBM, not the Infinity Cache)",
        "config": {"model": "c1: causal self-attention forward, fp32, B=32 H=8 S=256 D=32 (E=256), "
                            "no probs output", "global_batch": 32, "seq_len": 256, "B": 32, "H": 8, "S": 256, "D": 32,
                   "parallelism": "single GPU"},
    }
    if "us_per_call" in head:
        flops, _ = work(CONFIGS["c1"])
        ach = flops / (head["us_per_call"] * 1e-6)
        line["roofline"] = {
            "bound": "mfma", "achieved": round(ach / 1e12, 3), "peak": PEAK_F32_MFMA / 1e12,
            "unit": "TFLOP/s", "frac": round(ach / PEAK_F32_MFMA, 4),
            "frac_of_fp32_mfma": round(ach / RATE_F32_MFMA, 4), "traffic": read_traffic("c1"),
        }
    if cpu is not None:
        _, ncores, cfgs = cpu
        c1 = cfgs["c1"]["one_thread"]
        line["cpu_baseline"] = {
            "value": round(c1["gflops"] / 1e3, 6), "unit": "TFLOP/s", "cores": 1, "kind": "port",
            "sample": f"c1 through the oracle's scalar restatement of flash_attention_kernel<32>: {c1['pairs']} of "
                      f"{c1['of_pairs']} (b,h) pairs, median of {c1['runs']} runs on 1 thread, "
                      f"{c1['us_per_call']:.0f} us per call",
            "all_cores": {"value": round(cfgs["c1"]["all_cores"]["gflops"] / 1e3, 6), "cores": ncores,
                          "us_per_call": cfgs["c1"]["all_cores"]["us_per_call"]},
        }
    line["configs"] = {n: [round(r["us_per_call"], 2), round(r["roofline_frac"], 3)] if "us_per_call" in r
                       else "error: " + r.get("error", "")[:40] for n, r in results.items()}
    return line


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--only", default="", help="comma-separated config names (default: all)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the host baseline")
    ap.add_argument("--no-hot", action="store_true", help="skip the one-set (cache-hot) timing")
    ap.add_argument("--no-dist", action="store_true", help="skip the per-call distribution")
    ap.add_argument("--details", default="", help="file for everything measured (JSON)")
    ap.add_argument("--copy-mb", type=int, default=0,
                    help="also run one plain device copy of this many MiB (counter calibration)")
    args = ap.parse_args()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py: this build measures one MI355X only; the attention forward shards "
              "over (batch, head) with no exchange, so N GPUs run N independent copies.",
              file=sys.stderr)
        sys.exit(2)

    import torch

    from hipgpt_amd import attention as A

    dev = torch.device("cuda:0")
    names = [n for n in args.only.split(",") if n] or list(CONFIGS)
    unknown = [n for n in names if n not in CONFIGS]
    if unknown:
        sys.exit(f"bench.py: unknown config(s) {unknown}")
    results = {}
    # Bring the GPU to its steady clock before the first timed config.
    fn0, _ = make_call(CONFIGS[names[0]], torch, A, dev)
    t_end = time.perf_counter() + 0.5
    while time.perf_counter() < t_end:
        for _ in range(20):
            fn0()
        torch.cuda.synchronize()
    del fn0
    for name in names:
        cfg = CONFIGS[name]
        nsets = max(1, math.ceil(ROTATE_BYTES / set_bytes(cfg)))
        try:
            sets = [make_call(cfg, torch, A, dev, seed=SEED + i) for i in range(nsets)]
        except Exception as e:  # e.g. a dtype this build has no kernel for
            results[name] = {"error": str(e)}
            continue
        fns = [f for f, _ in sets]
        extra = sets[0][1]
        try:
            ms = time_call(fns, args.steps, args.warmup, torch)
            ms_hot = None if args.no_hot else time_call(fns[:1], args.steps, args.warmup, torch)
            dist = None if args.no_dist else launch_dist(fns, max(args.steps, 100), torch)
        except Exception as e:
            results[name] = {"error": str(e)}
            continue
        del sets, fns
        flops, nbytes = work(cfg)
        B, H, Sq, Sk, D, causal, dtype, probs, kind = cfg
        peak = PEAK_BF16_MFMA if dtype == "bf16" else PEAK_F32_MFMA
        t_mfma = flops / peak
        t_hbm = nbytes / PEAK_HBM
        bound = "hbm" if t_hbm > t_mfma else "mfma"
        tflops = flops / (ms * 1e-3) / 1e12
        gbs = nbytes / (ms * 1e-3) / 1e9
        frac = (t_hbm if bound == "hbm" else t_mfma) / (ms * 1e-3)
        results[name] = {
            "shape": {"B": B, "H": H, "Sq": Sq, "Sk": Sk, "D": D}, "causal": causal,
            "dtype": dtype, "probs": probs, "us_per_call": round(ms * 1e3, 3),
            "us_per_call_hot": None if ms_hot is None else round(ms_hot * 1e3, 3), "dist_us": dist,
            "sets": nsets, "tflops": round(tflops, 3), "gbs": round(gbs, 1), "bound": bound,
            "roofline_frac": round(frac, 4), **extra,
        }
        hot = "" if ms_hot is None else f" (hot {ms_hot * 1e3:.2f})"
        print(f"# {name}: {ms * 1e3:.2f} us{hot}  {tflops:.2f} TFLOP/s  {gbs:.0f} GB/s  "
              f"{bound}-bound frac {frac:.3f}  sets {nsets}", file=sys.stderr, flush=True)
        torch.cuda.empty_cache()

    if args.copy_mb > 0:
        # A plain copy of known size, for scaling FETCH_SIZE / WRITE_SIZE counters.
        n = args.copy_mb * (1 << 20) // 4
        src = torch.ones(n, device=dev)
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    cpu = None if args.no_cpu else cpu_baseline()
    if args.details:
        with open(args.details, "w") as f:
            json.dump({"configs": results, "cpu_baseline": cpu and {"host": cpu[0], "configs": cpu[2]}}, f, indent=1)
    print(json.dumps(headline(args.steps, args.warmup, results, cpu)), flush=True)


if __name__ == "__main__":
    main()
