"""The work that programs have this framework do, as cases to measure.

``listed()`` names one case per path and size class, ``draw(rng)`` gives
further sizes of the same paths.  A case's ``kind`` says which calls it makes:

* ``dropin``      -- ``launch_multihead_attention``: HipGPT's forward launcher
  (planar ``[Q|K|V]``, no mask, probs written).
* ``layer``       -- HipGPT's attention block: QKV projection, the launcher on
  its ``[T, 3E]`` buffer, output projection.
* ``causal``      -- ``qkv_planar`` with a causal mask and no probs.
* ``bf16``        -- ``attention`` on bf16 views of a packed ``[B, S, 3, H, D]``.
* ``prefill``     -- ``attention`` of a chunk of new queries against a longer
  key/value cache (causal, ``Sk >= Sq``), fp32.
* ``bwd_dropin``  -- ``launch_multihead_attention_backward`` on stored probs.
* ``bwd_causal``  -- ``attention_backward`` on causal stored probs.
* ``train``       -- ``fwd_lse_qkv_planar`` + ``bwd_lse_qkv_planar``, the
  training pair without a probs buffer.
* ``kvcache``     -- ``decode_kvcache``: one generation step over sequences of
  different lengths.
* ``projection``  -- ``qkv_projection`` into the planar buffer.
"""
import math

import torch

from hipgpt_amd import attention as A
from hipgpt_amd import projection as P


def listed():
    return [
        # HipGPT's generation call: one sequence, its default head shape
        {"name": "generate_b1", "kind": "dropin", "B": 1, "S": 256, "H": 8, "D": 32},
        # HipGPT's default model, one layer's attention block of a training batch
        {"name": "layer_default", "kind": "layer", "B": 32, "S": 256, "H": 8, "D": 32},
        # the same head shape through the causal entry point
        {"name": "causal_default", "kind": "causal", "B": 32, "S": 256, "H": 8, "D": 32},
        # a GPT-2-small layer's attention at its full context
        {"name": "causal_gpt2", "kind": "causal", "B": 8, "S": 1024, "H": 12, "D": 64},
        # the same layer fed by a bf16 projection
        {"name": "bf16_gpt2", "kind": "bf16", "B": 8, "S": 1024, "H": 12, "D": 64},
        # long rows at the larger head dim
        {"name": "causal_d128", "kind": "causal", "B": 4, "S": 2048, "H": 16, "D": 128},
        # a chunk of a prompt against what is cached of it, sizes as they come
        {"name": "prefill_ragged", "kind": "prefill", "B": 3, "S": 333, "Sk": 1357, "H": 12, "D": 64},
        # HipGPT's default model, the attention backward of a training batch
        {"name": "bwd_default", "kind": "bwd_dropin", "B": 32, "S": 256, "H": 8, "D": 32},
        # a GPT-2-small layer's attention in training, forward and backward
        {"name": "train_gpt2", "kind": "train", "B": 8, "S": 1024, "H": 12, "D": 64},
        # backward on stored causal probs at the larger head dim, odd length
        {"name": "bwd_d128_ragged", "kind": "bwd_causal", "B": 2, "S": 999, "H": 8, "D": 128},
        # one generation step of a batch of sequences that differ in length
        {"name": "kvcache_step", "kind": "kvcache", "B": 16, "S": 2048, "H": 12, "D": 64},
        # a GPT-2-small layer's QKV projection
        {"name": "projection_gpt2", "kind": "projection", "B": 8, "S": 1024, "H": 12, "D": 64},
    ]


# The most that a drawn case may ask for, per kind: (flops, elements of its
# largest tensor).
_LIMIT = {
    "dropin": (2.0e10, 5.5e7),
    "layer": (2.0e10, 2.0e7),
    "causal": (6.0e10, 5.0e7),
    "bf16": (6.0e10, 5.0e7),
    "prefill": (2.5e10, 5.0e7),
    "bwd_dropin": (1.5e10, 4.0e7),
    "bwd_causal": (1.5e10, 4.0e7),
    "train": (4.0e10, 4.0e7),
    "kvcache": (1.0e9, 3.0e7),
    "projection": (3.0e10, 3.0e7),
}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _largest(case):
    B, S, H, D = (case[k] for k in ("B", "S", "H", "D"))
    n = 3 * B * S * H * D
    if case["kind"] in ("dropin", "layer", "bwd_dropin", "bwd_causal"):
        n = max(n, B * H * S * S)
    if case["kind"] in ("prefill",):
        n = max(n, B * case["Sk"] * H * D)
    if case["kind"] == "kvcache":
        n = B * S * H * D
    return n


def draw(rng):
    while True:
        kind = rng.choice(sorted(_LIMIT))
        heads = {"bf16": [32, 64, 128], "layer": [32, 32, 64], "kvcache": [32, 64, 64, 128],
                 "train": [32, 64, 64, 80, 128], "causal": [32, 64, 64, 80, 128, 256],
                 "dropin": [32, 32, 64, 64, 96, 128]}
        case = {"kind": kind, "B": _log_int(rng, 1, 64), "S": _log_int(rng, 64, 2048), "H": rng.randint(1, 16),
                "D": rng.choice(heads.get(kind, [32, 64, 64, 128]))}
        if rng.random() < 0.4:  # as many lengths are whole tiles as are not
            case["S"] = max(64, case["S"] // 64 * 64)
        if kind == "prefill":
            case["Sk"] = case["S"] + _log_int(rng, 1, 2048)
        if work(case)["flops"] <= _LIMIT[kind][0] and _largest(case) <= _LIMIT[kind][1]:
            return case


# ------------------------------------------------------------------ inputs


def _rand(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return lambda *shape: torch.randn(*shape, device="cuda", generator=g)


def _heads(planar, B, S, H, D):
    """[3, B, H, S, D] in 64 bits of a flat planar [Q|K|V] buffer."""
    return planar.reshape(3, B, S, H, D).permute(0, 1, 3, 2, 4).contiguous().double()


def _softmax64(q, k, causal):
    """Probs and row log-sum-exp, in 64 bits, of [B, H, S, D] tensors."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    if causal:
        Sq, Sk = s.shape[-2:]
        s.masked_fill_(torch.ones(Sq, Sk, dtype=torch.bool, device=s.device).triu_(1 + Sk - Sq), -math.inf)
    lse = torch.logsumexp(s, -1)
    return s.sub_(lse.unsqueeze(-1)).exp_(), lse


def _rows(x):
    """[B, H, S, D] -> [B*S, H*D]"""
    B, H, S, D = x.shape
    return x.permute(0, 2, 1, 3).reshape(B * S, H * D)


def _attend64(q, k, v, causal):
    """Output and lse one sequence at a time (the probs of all would not fit)."""
    o, lse = torch.empty_like(q), torch.empty(q.shape[:-1], dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        p, lse[b] = _softmax64(q[b:b + 1], k[b:b + 1], causal)
        o[b:b + 1] = torch.matmul(p, v[b:b + 1])
    return o, lse


def _backward64(q, k, v, p, go):
    """dQ, dK, dV of softmax attention from its probs."""
    scale = q.shape[-1] ** -0.5
    dv = torch.matmul(p.transpose(-1, -2).contiguous(), go)
    dp = torch.matmul(go, v.transpose(-1, -2).contiguous())
    ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
    return torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2).contiguous(), q), dv


def _inputs(case, seed):
    """The tensors of a case, from the seed alone.  Queries, keys and values
    have unit variance, as a layer norm and a projection of unit gain leave
    them; gradients are small, as a mean loss makes them."""
    kind, B, S, H, D = (case[k] for k in ("kind", "B", "S", "H", "D"))
    E, T = H * D, B * S
    rand = _rand(seed)
    if kind in ("dropin", "causal"):
        return {"qkv": rand(3 * T * E)}
    if kind in ("layer", "projection"):
        t = {"x": rand(T, E), "w_qkv": rand(E, 3 * E) * E ** -0.5, "b_qkv": rand(3 * E) * 0.1}
        if kind == "layer":
            t.update(w_out=rand(E, E) * E ** -0.5, b_out=rand(E) * 0.1)
        return t
    if kind == "bf16":
        return {"qkv": rand(B, S, 3, H, D).bfloat16()}
    if kind == "prefill":
        return {"qkv": rand(B, S, 3, H, D), "cache": rand(2, B, case["Sk"], H, D)}
    if kind in ("bwd_dropin", "bwd_causal"):
        qkv = rand(3 * T * E)
        probs = torch.empty(B, H, S, S, device="cuda")
        q, k, _ = _heads(qkv, B, S, H, D)
        for b in range(B):
            probs[b] = _softmax64(q[b], k[b], kind == "bwd_causal")[0]
        return {"qkv": qkv, "grad_out": rand(T * E) * 1e-2, "probs": probs}
    if kind == "train":
        return {"qkv": rand(3 * T * E), "grad_out": rand(T * E) * 1e-2}
    assert kind == "kvcache"
    t = {"new": rand(B, 3, H, D), "cache": rand(2, B, S, H, D)}
    g = torch.Generator().manual_seed(seed)
    t["lens"] = torch.randint(S // 4, S, (B,), generator=g, dtype=torch.int32).cuda()
    return t


def prepare(case, seed):
    kind, B, S, H, D = (case[k] for k in ("kind", "B", "S", "H", "D"))
    E, T = H * D, B * S

    def buf(*shape):
        return torch.empty(*shape, device="cuda")

    st = dict(case, E=E, T=T, **_inputs(case, seed))
    if kind in ("dropin", "layer"):
        st.update(out=buf(T, E), probs=buf(B, H, S, S))
        if kind == "layer":
            st.update(qkv=buf(T * 3 * E), y=buf(T, E))
    elif kind == "causal":
        st.update(out=buf(T, E))
    elif kind in ("bf16", "prefill"):
        st.update(out=buf(B, S, H, D))
    elif kind in ("bwd_dropin", "bwd_causal"):
        st.update(grad=buf(3 * T * E), workspace=buf(B * H * S))
    elif kind == "train":
        st.update(out=buf(T, E), lse=buf(B, H, S), grad=buf(3 * T * E), workspace=buf(B * H * S))
    elif kind == "kvcache":
        ns = A.decode_default_splits(B, H, S)
        st.update(out=buf(B, H, D), splits=ns, workspace=buf(max(1, A.decode_workspace_bytes(B, H, D, ns) // 4)))
    else:
        st.update(qkv=buf(3, T, E))
    return st


# -------------------------------------------------------------------- calls


def run(st):
    kind, B, S, H, D, E, T = (st[k] for k in ("kind", "B", "S", "H", "D", "E", "T"))
    if kind == "dropin":
        A.launch_multihead_attention(st["qkv"], st["out"], st["probs"], B, S, E, H)
        return st["out"], st["probs"]
    if kind == "layer":
        P.launch_matmul_add_bias(st["x"], st["w_qkv"], st["b_qkv"], st["qkv"], T, E, 3 * E)
        A.launch_multihead_attention(st["qkv"], st["out"], st["probs"], B, S, E, H)
        P.launch_matmul_add_bias(st["out"], st["w_out"], st["b_out"], st["y"], T, E, E)
        return st["qkv"], st["out"], st["probs"], st["y"]
    if kind == "causal":
        A.qkv_planar(st["qkv"], st["out"], None, B, S, E, H, causal=True)
        return st["out"]
    if kind == "bf16":
        q, k, v = st["qkv"].unbind(2)
        return A.attention(q, k, v, out=st["out"], causal=True)
    if kind == "prefill":
        return A.attention(st["qkv"][:, :, 0], st["cache"][0], st["cache"][1], out=st["out"], causal=True)
    if kind == "bwd_dropin":
        A.launch_multihead_attention_backward(st["grad_out"], st["qkv"], st["probs"], st["grad"], B, S, E, H)
        return st["grad"]
    if kind == "bwd_causal":
        return A.attention_backward(st["grad_out"], st["qkv"], st["probs"], st["grad"], B, S, E, H, causal=True,
                                    workspace=st["workspace"])
    if kind == "train":
        A.fwd_lse_qkv_planar(st["qkv"], st["out"], st["lse"], B, S, E, H, causal=True)
        A.bwd_lse_qkv_planar(st["grad_out"], st["qkv"], st["out"], st["lse"], st["grad"], B, S, E, H, causal=True,
                             workspace=st["workspace"])
        return st["out"], st["lse"], st["grad"]
    if kind == "kvcache":
        # not the last layer of the step: the lengths advance there
        A.decode_kvcache(st["new"][:, 0], st["new"][:, 1], st["new"][:, 2], st["cache"][0], st["cache"][1],
                         st["lens"], out=st["out"], advance=False, num_splits=st["splits"],
                         workspace=st["workspace"])
        return st["out"], st["cache"][0], st["cache"][1]
    P.qkv_projection(st["x"], st["w_qkv"], st["b_qkv"], out=st["qkv"], planar=True)
    return st["qkv"]


def exact(case, seed):
    """What ``run`` returns, in 64 bits."""
    kind, B, S, H, D = (case[k] for k in ("kind", "B", "S", "H", "D"))
    E, T = H * D, B * S
    t = _inputs(case, seed)

    def launcher(planar):
        q, k, v = _heads(planar, B, S, H, D)
        p, o = torch.empty(B, H, S, S, dtype=torch.float64, device="cuda"), torch.empty_like(q)
        for b in range(B):
            p[b], _ = _softmax64(q[b], k[b], False)
            o[b] = torch.matmul(p[b], v[b])
        return _rows(o), p

    if kind == "dropin":
        return launcher(t["qkv"])
    if kind == "layer":
        qkv = t["x"].double() @ t["w_qkv"].double() + t["b_qkv"].double()
        o, p = launcher(qkv)
        return qkv.reshape(-1), o, p, o @ t["w_out"].double() + t["b_out"].double()
    if kind == "causal":
        return _rows(_attend64(*_heads(t["qkv"], B, S, H, D), True)[0])
    if kind in ("bf16", "prefill"):
        q, k, v = t["qkv"].unbind(2)
        if kind == "prefill":
            k, v = t["cache"]
        q, k, v = (x.permute(0, 2, 1, 3).contiguous().double() for x in (q, k, v))
        return _attend64(q, k, v, True)[0].permute(0, 2, 1, 3).contiguous()
    if kind in ("bwd_dropin", "bwd_causal", "train"):
        q, k, v = _heads(t["qkv"], B, S, H, D)
        go = _heads(t["grad_out"].repeat(3), B, S, H, D)[0]
        grad = torch.empty(3, B, H, S, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            p = t["probs"][b].double() if "probs" in t else _softmax64(q[b], k[b], True)[0]
            for i, d in enumerate(_backward64(q[b], k[b], v[b], p, go[b])):
                grad[i, b] = d
        grad = torch.cat([_rows(g).reshape(-1) for g in grad])
        if kind != "train":
            return grad
        o, lse = _attend64(q, k, v, True)
        return _rows(o), lse, grad
    if kind == "kvcache":
        kc, vc = t["cache"]
        out = torch.empty(B, H, D, dtype=torch.float64, device="cuda")
        for b, n in enumerate(t["lens"].tolist()):
            kc[b, n], vc[b, n] = t["new"][b, 1], t["new"][b, 2]
            q, k, v = (x.permute(1, 0, 2).contiguous().double()
                       for x in (t["new"][b, 0].unsqueeze(0), kc[b, :n + 1], vc[b, :n + 1]))
            out[b] = torch.matmul(_softmax64(q, k, False)[0], v).squeeze(1)
        return out, kc.double(), vc.double()
    y = t["x"].double() @ t["w_qkv"].double() + t["b_qkv"].double()
    return y.reshape(T, 3, E).permute(1, 0, 2).contiguous()


# -------------------------------------------------------------------- costs


def work(case):
    """4 D flops per visible (query, key) pair forward, 8 D backward, 2 per
    product of a projection; each input read once and each output written
    once."""
    kind, B, S, H, D = (case[k] for k in ("kind", "B", "S", "H", "D"))
    E, T = H * D, B * S
    full, half = B * H * S * S, B * H * S * (S + 1) // 2
    if kind == "dropin":
        return {"flops": 4.0 * D * full, "bytes": 4 * (4 * T * E + full)}
    if kind == "layer":
        return {"flops": 4.0 * D * full + 8.0 * T * E * E,
                "bytes": 4 * ((T * E + 3 * E * E + 3 * E + 3 * T * E) + (4 * T * E + full)
                              + (T * E + E * E + E + T * E))}
    if kind == "causal":
        return {"flops": 4.0 * D * half, "bytes": 16 * T * E}
    if kind == "bf16":
        return {"flops": 4.0 * D * half, "bytes": (3 * 2 + 4) * T * E}
    if kind == "prefill":
        pairs = B * H * (S * case["Sk"] - S * (S - 1) // 2)
        return {"flops": 4.0 * D * pairs, "bytes": 4 * (2 * T * E + 2 * B * case["Sk"] * E)}
    if kind == "bwd_dropin":
        return {"flops": 8.0 * D * full, "bytes": 4 * (7 * T * E + full)}
    if kind == "bwd_causal":
        return {"flops": 8.0 * D * half, "bytes": 4 * (7 * T * E + half)}
    if kind == "train":
        return {"flops": 12.0 * D * half, "bytes": 4 * (4 * T * E + B * H * S) + 4 * (8 * T * E + B * H * S)}
    if kind == "kvcache":
        keys = B * 5 * S // 8  # lengths are spread evenly over S/4 .. S
        return {"flops": 4.0 * E * keys, "bytes": 4 * (2 * keys * E + 6 * B * E)}
    return {"flops": 6.0 * T * E * E, "bytes": 4 * (T * E + 3 * E * E + 3 * E + 3 * T * E)}


def tolerance(case):
    """About four times what the calls show against ``exact`` over the listed
    sizes and some forty drawn ones: 32-bit sums 8e-7 (largest 1.3e-5), bf16
    inputs with probs rounded to bf16 1.3e-3 (largest 2.6e-2)."""
    if case["kind"] == "bf16":
        return {"rel": 5e-3, "max": 1e-1}
    return {"rel": 3e-6, "max": 6e-5}
