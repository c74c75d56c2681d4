"""The work this framework is measured by, as cases: what a user's program asks of it.

Two kinds of user. A program on the ``pulsar_cuda`` op surface (the model's own forward and
backward in PyTorch) calls the fused ops of a layer, one token at a time or a training
micro-batch at a time. A program on the engine (``pulsar_engine``) prefills prompts, verifies
token blocks over its caches and generates. Every case runs the full-size model's widths;
the weights are random of the scales ``pulsar_engine.weights`` documents, made on the GPU in
the kernel format a loaded checkpoint has.

``exact`` restates the ops and the model in plain torch, in 64 bits.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "pulsar-300m_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from pulsar_engine.config import PulsarConfig  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
F64 = torch.float64
CFG = PulsarConfig()
D, H, HKV, HD = CFG.d_model, CFG.n_heads, CFG.n_kv_heads, CFG.head_dim
E, K, V, P, L = CFG.n_routed_experts, CFG.top_k, CFG.vocab_size, CFG.default_pulses, CFG.n_core
DE, DS, EPS = CFG.d_expert, CFG.d_shared, CFG.rms_eps


# --------------------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------------------

def listed():
    return [
        # One decoded token of each of 16 sequences through the dense ops of a layer (norm,
        # stem conv, q/k norm + RoPE, attention gate, SwiGLU): the smallest call, host cost
        # and launch latency.
        dict(name="dense_ops_16x1_bf16", kind="dense", batch=16, tokens=1, dtype="bf16",
             train=False),
        # The same ops, forward and backward, over the training micro-batch that the
        # benchmark's op table is quoted on.
        dict(name="dense_train_8x2048_bf16", kind="dense", batch=8, tokens=2048, dtype="bf16",
             train=True),
        # fp32 training step of a short ragged batch (parity runs, fine-tuning on odd lengths).
        dict(name="dense_train_3x777_fp32", kind="dense", batch=3, tokens=777, dtype="fp32",
             train=True),
        # The MoE ops (router top-k, slots, dispatch, SwiGLU, combine) of a ragged evaluation
        # batch, forward only.
        dict(name="moe_ops_517_bf16", kind="moe", rows=517, dtype="bf16", train=False),
        # The MoE ops of a training micro-batch, forward and backward.
        dict(name="moe_train_16384_bf16", kind="moe", rows=16384, dtype="bf16", train=True),
        # One interactive prompt of odd length: time to first token.
        dict(name="prefill_1x517_bf16", kind="prefill", batch=1, prompt=517, dtype="bf16"),
        # The headline batch's prompts.
        dict(name="prefill_16x2048_bf16", kind="prefill", batch=16, prompt=2048, dtype="bf16"),
        # A single fp32 request end to end: prefill, then 64 tokens of the reference schedule.
        dict(name="generate_1x128_fp32", kind="generate", batch=1, prompt=128, new=64, draft=0,
             dtype="fp32"),
        # Decode of the headline batch: drafts of 4, sampled, 64 tokens each.
        dict(name="decode_16x2048_draft4_bf16", kind="decode", batch=16, prompt=2048, new=64,
             draft=4, dtype="bf16"),
        # Throughput serving: 256 short contexts, reference schedule, 32 tokens each.
        dict(name="decode_256x512_bf16", kind="decode", batch=256, prompt=512, new=32, draft=0,
             dtype="bf16"),
        # One forward pass of 4 long contexts (a token each) over the cache.
        dict(name="verify_4x32768_n1_bf16", kind="verify", batch=4, ctx=32768, n=1,
             dtype="bf16"),
        # The verify step: a 5-token block of each of 64 sequences over 8192 positions.
        dict(name="verify_64x8192_n5_bf16", kind="verify", batch=64, ctx=8192, n=5,
             dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "moe", "moe", "prefill", "prefill", "generate",
                       "decode", "verify", "verify"])
    half = rng.random() < 0.75
    if kind == "dense":
        batch = _log_int(rng, 1, 16)
        return dict(kind=kind, batch=batch, tokens=_log_int(rng, 1, 16384 // batch),
                    dtype="bf16" if half else "fp32", train=rng.random() < 0.6)
    if kind == "moe":
        return dict(kind=kind, rows=_log_int(rng, 1, 16384), dtype="bf16" if half else "fp32",
                    train=rng.random() < 0.6)
    if kind == "prefill":
        if not half:
            return dict(kind=kind, batch=rng.randint(1, 2), prompt=_log_int(rng, 1, 300),
                        dtype="fp32")
        batch = _log_int(rng, 1, 16)
        return dict(kind=kind, batch=batch, prompt=_log_int(rng, 1, min(4096, 32768 // batch)),
                    dtype="bf16")
    if kind == "generate":
        if not half:
            return dict(kind=kind, batch=1, prompt=_log_int(rng, 2, 128),
                        new=_log_int(rng, 4, 64), draft=rng.choice([0, 4]), dtype="fp32")
        return dict(kind=kind, batch=_log_int(rng, 1, 16), prompt=_log_int(rng, 2, 1024),
                    new=_log_int(rng, 4, 64), draft=rng.choice([0, 4, 6]), dtype="bf16")
    if kind == "decode":
        batch = _log_int(rng, 1, 256)
        return dict(kind=kind, batch=batch, prompt=_log_int(rng, 16, min(4096, 131072 // batch)),
                    new=_log_int(rng, 4, 32), draft=rng.choice([0, 4, 6]) if batch <= 64 else 0,
                    dtype="bf16")
    batch = _log_int(rng, 1, 128)
    return dict(kind=kind, batch=batch, ctx=_log_int(rng, 64, min(32768, 524288 // batch)),
                n=rng.randint(1, 8 if batch <= 64 else 4), dtype="bf16")


# --------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _tables(theta, n):
    """Angles of the rotary tables as the model defines them (fp32 products), [n, 32]."""
    inv = 1.0 / (theta ** (torch.arange(0, HD, 2, dtype=torch.float32) / HD))
    return torch.outer(torch.arange(n, dtype=torch.float32), inv).to(DEV)


def _dense_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    B, T = case["batch"], case["tokens"]
    ang = _tables(CFG.rope_theta_local, T)
    s = dict(x=_randn(g, B, T, D, dtype=dt), norm_w=1.0 + _randn(g, D, std=0.1),
             qkv=_randn(g, B, T, (H + 2 * HKV) * HD, dtype=dt),
             q_w=1.0 + _randn(g, H, HD, std=0.1), k_w=1.0 + _randn(g, HKV, HD, std=0.1),
             cos=ang.cos(), sin=ang.sin(), attn=_randn(g, B, H, T, HD, dtype=dt),
             gate=2.0 + _randn(g, B, T, H), conv_w=_randn(g, D, 4, std=0.3),
             gu=_randn(g, B, T, 2 * DS, dtype=dt))
    if case["train"]:
        s.update(d_y=_randn(g, B, T, D, dtype=dt), d_q=_randn(g, B, H, T, HD, dtype=dt),
                 d_k=_randn(g, B, HKV, T, HD, dtype=dt),
                 d_gated=_randn(g, B, T, H * HD, dtype=dt),
                 d_conv=_randn(g, B, T, D, dtype=dt), d_act=_randn(g, B, T, DS, dtype=dt))
    return s


def _capacity(n):
    return max(32, -(-math.ceil(n * K / E * CFG.moe_capacity_factor) // 32) * 32)


def _moe_inputs(case, seed):
    """The selection (idx, its order by expert and weight, slots) follows the logits, as the
    model computes it between these ops with torch's own sort."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    N = case["rows"]
    C = _capacity(N)
    logits, bias = _randn(g, N, E, std=0.64, dtype=dt), _randn(g, E, std=0.01)
    score = torch.sigmoid(logits.double() - logits.double().mean(1, keepdim=True))
    idx = (score + bias.double()).topk(K, dim=1).indices
    w = score.gather(1, idx)
    w = (w / (w.sum(1, keepdim=True) + 1e-6)).to(torch.bfloat16)
    flat = idx.reshape(-1).contiguous()
    wf = w.reshape(-1).float()
    order = torch.argsort(flat.float() - 0.5 * wf / (1.0 + wf), stable=True)
    rank = torch.empty_like(flat)
    start = torch.bincount(flat, minlength=E).cumsum(0) - torch.bincount(flat, minlength=E)
    rank[order] = torch.arange(N * K, device=DEV) - start[flat[order]]
    slots = torch.where(rank < C, rank, -1).to(torch.int32).view(N, K).contiguous()
    s = dict(x=_randn(g, N, D, dtype=dt), logits=logits, bias=bias, idx=idx.contiguous(), w=w,
             flat=flat, order=order, slots=slots, C=C,
             counts=torch.bincount(flat, minlength=E).clamp_max(C),
             gu=_randn(g, E, C, 2 * DE, dtype=dt), eo=_randn(g, E, C, D, dtype=dt),
             shared=_randn(g, N, D, dtype=dt))
    if case["train"]:
        s.update(d_out=_randn(g, N, D, dtype=dt), d_act=_randn(g, E, C, DE, dtype=dt),
                 d_in=_randn(g, E, C, D, dtype=dt),
                 d_w=_randn(g, N, K, dtype=torch.bfloat16), d_z=torch.ones((), device=DEV),
                 d_pm=_randn(g, E))
    return s


def _weights(seed, dt):
    """Plain [..., N, K] weights of the model. The output head is the embedding under a fixed
    permutation of the vocabulary: logits are then as peaked as a trained model's (a plain
    tied head on random weights repeats the current token for ever), and a stream is decided
    by more than its last bits."""
    g = _gen(seed)

    def n(*shape, std=0.02, t=dt):
        return _randn(g, *shape, std=std, dtype=t)

    f32 = torch.float32
    emb = n(V, D)
    w = dict(tok_emb=emb, lm_head=emb[torch.randperm(V, generator=g, device=DEV)],
             anchor_norm=1.0 + n(D, std=0.1, t=f32), state_norm=1.0 + n(D, std=0.1, t=f32),
             final_norm=1.0 + n(D, std=0.1, t=f32), step_emb=n(P, D),
             reinject_down=n(P, 8, 2 * D), reinject_up=n(P, D, 8),
             reinject_bias=n(P, D, std=0.1), res_scale=(1.0 + n(P, D, std=0.1, t=f32)).to(dt),
             conv_w=n(D, 4, t=f32))
    qkv = CFG.qkv_dim
    for i in range(L):
        w.update({f"layers.{i}.{k}": v for k, v in dict(
            attn_norm=1.0 + n(P, D, std=0.1, t=f32), mlp_norm=1.0 + n(P, D, std=0.1, t=f32),
            wqkvg=n(P, qkv + H, D), wo=n(P, D, H * HD),
            gate_bias=(2.0 + n(P, H, std=0.1, t=f32)).to(dt),
            q_norm=1.0 + n(P, H, HD, std=0.1, t=f32), k_norm=1.0 + n(P, HKV, HD, std=0.1, t=f32),
            v_lambda=torch.full((P,), 0.1, device=DEV).to(dt).float(),
            shared_gu=n(2 * DS, D), shared_down=n(D, DS), routed_gu=n(E, 2 * DE, D),
            routed_down=n(E, D, DE), router=n(P, E, D, t=f32),
            expert_bias=n(P, E, std=0.01, t=f32),
            routed_scale=(1.0 + n(P, D, std=0.1, t=f32)).to(dt)).items()})
    return w


_GEMM = ("lm_head", "wqkvg", "wo", "shared_gu", "shared_down", "routed_gu", "routed_down")


def _model(seed, dt):
    from pulsar_engine.model import DeviceModel, pack_mfma

    w = _weights(seed, dt)
    if dt == torch.bfloat16:
        for k in w:
            if k.split(".")[-1] in _GEMM:
                w[k] = pack_mfma(w[k])
    return DeviceModel(CFG, w, dt, device=DEV, kernel_format=True)


def _ids(seed, batch, n):
    """Token ids of Zipf frequencies, as text has them."""
    g = _gen(seed + 977)
    p = torch.arange(1, V + 1, device=DEV, dtype=F64) ** -1.1
    c = (p / p.sum()).cumsum(0)
    u = torch.rand(batch, n, generator=g, device=DEV, dtype=F64)
    return torch.searchsorted(c, u).clamp_max(V - 1).to(torch.int32).cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dense":
        return dict(case=case, **_dense_inputs(case, seed))
    if kind == "moe":
        return dict(case=case, **_moe_inputs(case, seed))
    from pulsar_engine.engine import HipEngine, PulsarInferenceEngine

    B, dt = case["batch"], DTYPES[case["dtype"]]
    model = _model(seed, dt)
    s = dict(case=case, model=model, seed=seed)
    if kind == "generate":
        s["engine"] = PulsarInferenceEngine(model)
        s["ids"] = _ids(seed, B, case["prompt"]).tolist()
        return s
    if kind == "prefill":
        s["engine"] = HipEngine(model, batch=B, max_prompt=case["prompt"], max_new=16,
                                temperature=0.0, stop_ids=[], seed=seed)
        s["ids"] = _ids(seed, B, case["prompt"])
        rows = B
    elif kind == "decode":
        # sampled, with the benchmark's settings
        s["engine"] = HipEngine(model, batch=B, max_prompt=case["prompt"], max_new=case["new"],
                                temperature=0.8, top_p=0.95, repetition_penalty=1.15,
                                stop_ids=[], seed=seed, draft_len=case["draft"])
        s["engine"].prefill(_ids(seed, B, case["prompt"]))
        rows = B
    else:
        n = case["n"]
        s["engine"] = HipEngine(model, batch=B, max_prompt=1, max_new=8, temperature=0.0,
                                stop_ids=[], draft_len=0 if n <= 2 else n - 1,
                                max_ctx=case["ctx"] + 16)
        s["engine"].fill_kv(case["ctx"], seed=seed)
        s["ids"] = _ids(seed, B, n)
        rows = B * n
    s["logits"] = torch.empty(rows, V, dtype=torch.float32, pin_memory=True)
    return s


# --------------------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------------------

def _run_dense(s):
    import pulsar_cuda as pc

    case = s["case"]
    T = case["tokens"]
    q = s["qkv"][..., : H * HD].view(case["batch"], T, H, HD).transpose(1, 2)
    k = s["qkv"][..., H * HD: (H + HKV) * HD].view(case["batch"], T, HKV, HD).transpose(1, 2)
    y, rs = pc.rmsnorm_forward(s["x"], s["norm_w"], EPS)
    conv = pc.causal_depthwise_conv1d_k4_forward(s["x"], s["conv_w"])
    qr, q_rs = pc.qk_rmsnorm_rope_forward(q, s["q_w"], s["cos"], s["sin"], T, EPS)
    kr, k_rs = pc.qk_rmsnorm_rope_forward(k, s["k_w"], s["cos"], s["sin"], T, EPS)
    gated = pc.fused_attn_gate_forward(s["attn"], s["gate"])
    act = pc.fused_swiglu_forward(s["gu"], DS)
    out = dict(y=y, rs=rs, conv=conv, q=qr, q_rs=q_rs, k=kr, k_rs=k_rs, gated=gated, act=act)
    if case["train"]:
        out["d_gu"] = pc.fused_swiglu_backward(s["d_act"], s["gu"], DS)
        out["d_attn"], out["d_gate"] = pc.fused_attn_gate_backward(s["d_gated"], s["attn"],
                                                                   s["gate"])
        out["d_k"], out["d_kw"] = pc.qk_rmsnorm_rope_backward(s["d_k"], k, s["k_w"], k_rs,
                                                              s["cos"], s["sin"], T)
        out["d_q"], out["d_qw"] = pc.qk_rmsnorm_rope_backward(s["d_q"], q, s["q_w"], q_rs,
                                                              s["cos"], s["sin"], T)
        out["d_xc"], out["d_cw"] = pc.causal_depthwise_conv1d_k4_backward(s["d_conv"], s["x"],
                                                                          s["conv_w"])
        out["d_x"], out["d_nw"] = pc.rmsnorm_backward(s["d_y"], s["x"], s["norm_w"], rs)
    return out


def _run_moe(s):
    import pulsar_cuda as pc

    case, C = s["case"], s["C"]
    N = case["rows"]
    idx, w, z, pm = pc.moe_router_topk_forward(s["logits"], s["bias"], K, 1e-3)
    slots, counts = pc.moe_slots_from_order(s["flat"], s["order"], E, C)
    ei = pc.moe_dispatch_forward(s["x"], s["idx"], s["slots"], E, C, s["counts"])[0]
    act = pc.fused_swiglu_forward(s["gu"], DE)
    y = pc.moe_combine_forward(s["eo"], s["idx"], s["w"], s["slots"], s["shared"])
    # dispatch writes slots below an expert's count and zeroes the rest: all of ei is written
    out = dict(idx=idx, w=w, z=z, pm=pm, slots=slots, counts=counts, ei=ei, act=act, y=y)
    if case["train"]:
        out["d_eo"], out["d_tw"] = pc.moe_combine_backward(s["d_out"], s["eo"], s["idx"], s["w"],
                                                           s["slots"], s["counts"])
        out["d_gu"] = pc.fused_swiglu_backward(s["d_act"], s["gu"], DE)
        out["d_x"] = pc.moe_dispatch_backward(s["d_in"], s["idx"], s["slots"], N, D)
        out["d_logits"] = pc.moe_router_topk_backward(s["d_w"], s["logits"], s["idx"], 1e-3,
                                                      s["d_z"], s["d_pm"])
    return out


def _logits(s):
    """The engine's logits, read into the program's own page-locked buffer."""
    from pulsar_cuda import _lib

    eng, buf = s["engine"], s["logits"]
    _lib.check(eng.lib.pulsar_engine_read(eng.handle, _lib.BUF_LOGITS, buf.data_ptr(),
                                          buf.numel() * 4,
                                          torch.cuda.current_stream().cuda_stream))
    return buf


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dense":
        return _run_dense(state)
    if kind == "moe":
        return _run_moe(state)
    eng = state["engine"]
    if kind == "generate":
        toks = eng.generate_ids(state["ids"], max_new_tokens=case["new"], temperature=0.0,
                                stop_ids=[], seed=0, draft_len=case["draft"])
        return dict(tokens=np.asarray(toks), logits=eng.last_engine.logits(case["batch"]))
    if kind == "prefill":
        eng.prefill(state["ids"])
        return dict(logits=_logits(state))
    if kind == "decode":
        eng.rewind(state["seed"])
        eng.run()
        return dict(tokens=np.asarray(eng.tokens()), logits=_logits(state))
    eng.verify(state["ids"], graph=True)
    return dict(logits=_logits(state))


# --------------------------------------------------------------------------------------
# Work, tolerance
# --------------------------------------------------------------------------------------

def _layer_weights(rows):
    """Weight elements one pass over `rows` rows needs of a layer."""
    hit = E * (1.0 - (1.0 - K / E) ** rows)
    return (CFG.qkv_dim + H) * D + D * H * HD + 3 * DS * D + hit * 3 * DE * D


_ROW_FLOPS = 2.0 * L * ((CFG.qkv_dim + H) * D + D * H * HD + 3 * DS * D + K * 3 * DE * D)


def _pass_bytes(es, rows, seqs, ctx):
    """One pulse over `rows` rows of `seqs` sequences with ctx cached positions each."""
    kv = 0
    for i in range(L):
        kv += 2 * HKV * HD * es * min(ctx, CFG.sliding_window if CFG.is_local(i) else ctx)
    return es * L * _layer_weights(rows) + seqs * kv


def work(case):
    es = 2 if case["dtype"] == "bf16" else 4
    kind = case["kind"]
    if kind == "dense":
        n = case["batch"] * case["tokens"]
        act = n * (2 * D + 2 * D + 2 * (H + HKV) * HD + 2 * H * HD + 3 * DS) - n * D
        b = act * es + n * (1 + H + HKV + H) * 4
        if case["train"]:
            # inputs of the backward, its own outputs
            b += es * n * (5 * DS + 3 * H * HD + 3 * (H + HKV) * HD + 3 * D + 3 * D)
            b += n * 4 * (2 * H + H + HKV + 1)
        return {"bytes": float(b), "flops": 40.0 * n * D}
    if kind == "moe":
        n, C = case["rows"], _capacity(case["rows"])
        kept = min(n * K, E * C)
        b = es * (n * E + n * D + E * C * D + 3 * E * C * DE + kept * D + 2 * n * D)
        b += n * K * (8 + 2 + 8 + 8 + 4 + 8 + 4 + 2 + 8 + 4 + 2)
        if case["train"]:
            b += es * (n * D + kept * D + E * C * D + 5 * E * C * DE + kept * D + n * D + 2 * n * E)
            b += n * K * (8 + 4 + 2 + 2 + 8 + 4 + 2 + 8)
        return {"bytes": float(b), "flops": 20.0 * n * K * D}
    B = case["batch"]
    head = es * V * D

    def prefill(T):
        n = B * T
        keys = sum((min(T, CFG.sliding_window) if CFG.is_local(i) else T) for i in range(L))
        att = sum(4.0 * H * HD * B * sum(min(t + 1, k) for t in range(T))
                  for k in [min(T, CFG.sliding_window) if CFG.is_local(i) else T
                            for i in range(L)])
        return (es * P * L * _layer_weights(n) + head + n * D * es + es * 2 * HKV * HD * B * keys,
                P * (n * _ROW_FLOPS + att) + 2.0 * B * V * D)

    if kind == "prefill":
        b, f = prefill(case["prompt"])
        return {"bytes": float(b + 4 * B * V), "flops": float(f)}
    if kind in ("generate", "decode"):
        b, f = prefill(case["prompt"]) if kind == "generate" else (0.0, 0.0)
        new, g, ctx = case["new"], case["draft"], case["prompt"] + case["new"] // 2
        if g == 0:  # an accepted token: two steps, one of them with logits
            b += new * (2 * _pass_bytes(es, B, B, ctx) + head)
        else:  # a round: g + 1 pulse-0 passes with g logits rows, the verify's other pulses
            r = new / (g + 1)
            b += r * ((g + 1) * _pass_bytes(es, B, B, ctx) + (g + 1) * head
                      + (P - 1) * _pass_bytes(es, B * (g + 1), B, ctx))
        att = 4.0 * H * HD * sum(min(ctx, CFG.sliding_window) if CFG.is_local(i) else ctx
                                 for i in range(L))
        f += B * new * (P * (_ROW_FLOPS + att) + 2.0 * 2 * V * D)
        return {"bytes": float(b + 4 * B * V), "flops": float(f)}
    n, ctx = case["n"], case["ctx"]
    att = 4.0 * H * HD * sum(min(ctx, CFG.sliding_window) if CFG.is_local(i) else ctx
                             for i in range(L))
    return {"bytes": float(P * _pass_bytes(es, B * n, B, ctx) + head + 4 * B * n * V),
            "flops": float(B * n * (P * (_ROW_FLOPS + att) + 2.0 * V * D))}


def tolerance(case):
    if case["kind"] in ("dense", "moe"):
        # one rounding to the storage type per output, fp32 sums for the weight gradients
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    # 24 layer passes with every activation stored in bf16 and a router whose near-ties fall
    # either way: 2.2e-2 to 2.7e-2 off the same model in 64 bits
    return {"rel": 3e-2}


# --------------------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------------------

def _rms(x, w, eps=EPS):
    r = torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return x * r * w, r


def _rope(x, c, s):
    a, b = x[..., : HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _shift(x, k):
    """x[:, t - k], zero before the start."""
    return torch.nn.functional.pad(x, (0, 0, k, 0))[:, : x.shape[1]] if k else x


def _swiglu(gu):
    g, u = gu.chunk(2, -1)
    return g * torch.sigmoid(g) * u


def _swiglu_back(d, gu):
    g, u = gu.chunk(2, -1)
    s = torch.sigmoid(g)
    return torch.cat([d * u * s * (1 + g * (1 - s)), d * g * s], -1)


def _exact_dense(case, seed):
    s = {k: v.double() for k, v in _dense_inputs(case, seed).items()}
    B, T = case["batch"], case["tokens"]
    q = s["qkv"][..., : H * HD].view(B, T, H, HD).transpose(1, 2)
    k = s["qkv"][..., H * HD: (H + HKV) * HD].view(B, T, HKV, HD).transpose(1, 2)
    y, rs = _rms(s["x"], s["norm_w"])
    conv = s["x"] + sum(s["conv_w"][:, j] * _shift(s["x"], j) for j in range(4))
    out = dict(y=y, rs=rs.reshape(-1), conv=conv)
    for n, v, w in (("q", q, s["q_w"]), ("k", k, s["k_w"])):
        nv, r = _rms(v, w[None, :, None])
        out[n], out[n + "_rs"] = _rope(nv, s["cos"], s["sin"]), r.reshape(-1)
    g = torch.sigmoid(s["gate"])
    out["gated"] = (s["attn"].transpose(1, 2) * g[..., None]).reshape(B, T, H * HD)
    out["act"] = _swiglu(s["gu"])
    if not case["train"]:
        return out
    out["d_gu"] = _swiglu_back(s["d_act"], s["gu"])
    dg = s["d_gated"].view(B, T, H, HD)
    out["d_attn"] = (dg * g[..., None]).transpose(1, 2)
    out["d_gate"] = (dg * s["attn"].transpose(1, 2)).sum(-1) * g * (1 - g)
    for n, v, w, d in (("k", k, s["k_w"], s["d_k"]), ("q", q, s["q_w"], s["d_q"])):
        r = torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + EPS)
        dn = _rope(d, s["cos"], -s["sin"])
        wv = w[None, :, None]
        out["d_" + n] = r * wv * dn - v * r ** 3 * (dn * v * wv).sum(-1, keepdim=True) / HD
        out["d_" + n + "w"] = (dn * v * r).sum((0, 2))
    d = s["d_conv"]
    ahead = [torch.nn.functional.pad(d, (0, 0, 0, j))[:, j:] for j in range(4)]
    out["d_xc"] = d + sum(s["conv_w"][:, j] * ahead[j] for j in range(4))
    out["d_cw"] = torch.stack([(d * _shift(s["x"], j)).sum((0, 1)) for j in range(4)], 1)
    r, x, w, d = rs, s["x"], s["norm_w"], s["d_y"]
    out["d_x"] = r * w * d - x * r ** 3 * (d * x * w).sum(-1, keepdim=True) / D
    out["d_nw"] = (d * x * r).sum((0, 1))
    return out


def _exact_moe(case, seed):
    s = _moe_inputs(case, seed)
    N, C = case["rows"], s["C"]
    lg = s["logits"].double()
    c = lg - lg.mean(1, keepdim=True)
    sc, lse = torch.sigmoid(c), torch.logsumexp(c, 1)
    idx = (sc + s["bias"].double()).topk(K, dim=1).indices
    u = sc.gather(1, idx)
    den = u.sum(1, keepdim=True) + 1e-6
    kept = s["slots"] >= 0
    at = s["idx"] * C + s["slots"].clamp_min(0)
    rows = torch.arange(N, device=DEV)[:, None].expand(N, K)
    ei = torch.zeros(E * C, D, dtype=F64, device=DEV)
    ei[at[kept]] = s["x"].double()[rows[kept]]
    eo, wts = s["eo"].double().view(E * C, D), s["w"].double()
    y = s["shared"].double()
    for j in range(K):
        y = y + (wts[:, j] * kept[:, j])[:, None] * eo[at[:, j]]
    out = dict(idx=idx, w=u / den, z=1e-3 * lse.pow(2).mean(), pm=sc.mean(0),
               slots=s["slots"].reshape(-1),
               counts=torch.bincount(s["flat"], minlength=E), ei=ei.view(E, C, D),
               act=_swiglu(s["gu"].double()), y=y)
    if not case["train"]:
        return out
    d = s["d_out"].double()
    deo = torch.zeros(E * C, D, dtype=F64, device=DEV)
    deo[at[kept]] = wts[kept][:, None] * d[rows[kept]]
    out["d_eo"] = deo.view(E, C, D)
    out["d_tw"] = torch.stack([(d * eo[at[:, j]]).sum(1) * kept[:, j] for j in range(K)], 1)
    out["d_gu"] = _swiglu_back(s["d_act"].double(), s["gu"].double())
    din = s["d_in"].double().view(E * C, D)
    out["d_x"] = sum(din[at[:, j]] * kept[:, j, None] for j in range(K))
    u = sc.gather(1, s["idx"])
    den = u.sum(1, keepdim=True) + 1e-6
    dw = s["d_w"].double()
    g = 2e-3 * lse[:, None] * torch.softmax(c, 1) / N + s["d_pm"].double() / N * sc * (1 - sc)
    g = g.scatter_add(1, s["idx"], (dw - (dw * u).sum(1, keepdim=True) / den) / den * u * (1 - u))
    out["d_logits"] = g - g.mean(1, keepdim=True)
    return out


class _Net:
    """The model in 64 bits: passes over [B, n, D] rows."""

    def __init__(self, seed, dt):
        self.w = _weights(seed, dt)
        self.rope = {}

    def t(self, name, *at):
        v = self.w[name]
        for i in at:
            v = v[i]
        return v.double()

    def angles(self, local, pos):
        ang = _tables(CFG.rope_theta_local if local else CFG.rope_theta_global, pos[-1] + 1)
        ang = ang[pos[0]:].double()
        return ang.cos(), ang.sin()

    def pulse_input(self, k, e, prev):
        if k == 0:
            return e + self.t("step_emb", 0)
        r = _rms(prev, self.t("state_norm"))[0]
        g = torch.cat([e, r], -1) @ self.t("reinject_down", k).T
        mix = torch.sigmoid(g @ self.t("reinject_up", k).T + self.t("reinject_bias", k))
        return r + mix * (e - r) + self.t("step_emb", k)

    def moe(self, i, k, x, capacity):
        """x [B, n, D]; capacity None: every assignment kept, else per sequence and expert."""
        B, n, _ = x.shape
        f = x.reshape(-1, D)
        lw = f"layers.{i}."
        lg = f @ self.t(lw + "router", k).T
        sc = torch.sigmoid(lg - lg.mean(1, keepdim=True))
        idx = (sc + self.t(lw + "expert_bias", k)).topk(K, 1).indices
        w = sc.gather(1, idx)
        w = w / (w.sum(1, keepdim=True) + 1e-6)
        if capacity is not None:
            for b in range(B):
                for e in range(E):
                    sel = idx[b * n:(b + 1) * n] == e
                    if int(sel.sum()) > capacity:
                        wb = torch.where(sel, w[b * n:(b + 1) * n], -1.0).reshape(-1)
                        drop = torch.argsort(wb, descending=True, stable=True)[capacity:]
                        drop = drop[sel.reshape(-1)[drop]]
                        w[b * n:(b + 1) * n].view(-1)[drop] = 0.0
        out = _swiglu(f @ self.t(lw + "shared_gu").T) @ self.t(lw + "shared_down").T
        routed = torch.zeros_like(f)
        for e in range(E):
            r, j = (idx == e).nonzero(as_tuple=True)
            if len(r):
                a = _swiglu(f[r] @ self.t(lw + "routed_gu", e).T)
                routed.index_add_(0, r, (a @ self.t(lw + "routed_down", e).T) * w[r, j, None])
        return (out + routed * self.t(lw + "routed_scale", k)).view(B, n, D)

    def layer(self, i, k, h, pos, v_first, attend, capacity, yarn):
        B, n, _ = h.shape
        lw, local = f"layers.{i}.", CFG.is_local(i)
        x = _rms(h, self.t(lw + "attn_norm", k))[0]
        y = x @ self.t(lw + "wqkvg", k).T
        q = y[..., : H * HD].view(B, n, H, HD).transpose(1, 2)
        kk = y[..., H * HD:(H + HKV) * HD].view(B, n, HKV, HD).transpose(1, 2)
        v = y[..., (H + HKV) * HD: CFG.qkv_dim].view(B, n, HKV, HD).transpose(1, 2)
        gate = torch.sigmoid(y[..., CFG.qkv_dim:] + self.t(lw + "gate_bias", k))
        if i == 0 and k == 0:
            v_first = v
        elif v_first is not None:
            lam = self.t(lw + "v_lambda", k)
            v = (1 - lam) * v + lam * v_first
        c, s = self.angles(local, pos)
        q = _rope(_rms(q, self.t(lw + "q_norm", k)[:, None])[0], c, s)
        kk = _rope(_rms(kk, self.t(lw + "k_norm", k)[:, None])[0], c, s)
        if yarn and not local:
            p = torch.arange(pos[0], pos[-1] + 1, device=DEV, dtype=F64) + 1
            q = q * (1 + 0.1 * torch.log(p.clamp_min(CFG.base_seq_len) / CFG.base_seq_len))[:, None]
        a = attend(i, local, q, kk, v)
        a = a.transpose(1, 2) * gate[..., None]
        h = h + a.reshape(B, n, H * HD) @ self.t(lw + "wo", k).T
        return h + self.moe(i, k, _rms(h, self.t(lw + "mlp_norm", k))[0], capacity), v_first

    def pulses(self, e, pos, attend, capacity, yarn):
        h = None
        for k in range(P):
            h_in = self.pulse_input(k, e, h)
            h, v_first = h_in, None
            for i in range(L):
                h, v_first = self.layer(i, k, h, pos, v_first, attend, capacity, yarn)
            h = h_in + (h - h_in) * self.t("res_scale", k)
        return h

    def head(self, h):
        return _rms(h, self.t("final_norm"))[0] @ self.t("lm_head").T


def _sdpa(q, k, v, mask):
    """q [H, n, 64], k and v [HKV, S, 64], mask [n, S] (True: attended)."""
    q = q.view(HKV, -1, HD)  # the four query heads of a KV head
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / 8.0
    s = s.view(HKV, H // HKV, -1, k.shape[1]).masked_fill(~mask, -math.inf)
    return torch.matmul(torch.softmax(s, -1).view(HKV, -1, k.shape[1]), v).view(H, -1, HD)


def _exact_prefill(case, seed):
    net, T, W = _Net(seed, DTYPES[case["dtype"]]), case["prompt"], CFG.sliding_window
    ids = torch.from_numpy(_ids(seed, case["batch"], T)).to(DEV).long()

    def attend(i, local, q, k, v):
        # a sliding-window layer keeps the last W keys of the prompt and masks them from its
        # first key on, whatever position the query has
        if local and T > W:
            k, v = k[:, :, -W:], v[:, :, -W:]
        t, j = torch.arange(T, device=DEV), torch.arange(k.shape[2], device=DEV)
        out = torch.empty_like(q)
        for b in range(q.shape[0]):
            for lo in range(0, T, 2048):
                sl = slice(lo, min(T, lo + 2048))
                out[b, :, sl] = _sdpa(q[b, :, sl].contiguous(), k[b], v[b], j <= t[sl, None])
        return out

    a = _rms(net.t("tok_emb")[ids], net.t("anchor_norm"))[0]
    e = a + sum(net.t("conv_w")[:, j] * _shift(a, j) for j in range(4))
    h = net.pulses(e, range(T), attend, _capacity(T), False)
    return dict(logits=net.head(h[:, -1]))


def _mix64(z):
    def shr(x, n):
        return (x >> n) & ((1 << (64 - n)) - 1)

    z = (z ^ shr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ shr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ shr(z, 31)


def _cached(seed, layer, which, index, dt):
    """Elements of the synthetic cache: N(0, 1) by Box-Muller from a counter."""
    sd = _mix64(torch.tensor([seed ^ (2 * layer + which + 1)], dtype=torch.int64, device=DEV))
    h = _mix64(sd + (0x9E3779B97F4A7C15 - (1 << 64)) * (index + 1))
    u1 = (((h >> 40) & 0xFFFFFF) + 1).double() / 16777216.0
    u2 = ((h >> 16) & 0xFFFFFF).double() / 16777216.0
    return (torch.sqrt(-2 * torch.log(u1)) * torch.cos(2 * math.pi * u2)).to(dt).double()


def _exact_verify(case, seed):
    B, n, ctx, W = case["batch"], case["n"], case["ctx"], CFG.sliding_window
    dt = DTYPES[case["dtype"]]
    net = _Net(seed, dt)
    ids = torch.from_numpy(_ids(seed, B, n)).to(DEV).long()
    lcap, pages = (W + 8 + 63) // 64 * 64, (ctx + 16 + 63) // 64
    g = torch.arange(HKV, device=DEV)[:, None, None]
    d = torch.arange(HD, device=DEV)[None, None, :]
    cache = {}

    def cached(i, local, b):
        if (i, b) not in cache:
            pos = torch.arange(max(0, ctx - W) if local else 0, ctx, device=DEV)[None, :, None]
            if local:
                at = ((b * HKV + g) * lcap + pos % lcap) * HD + d
                av = ((b * HKV + g) * HD + d) * lcap + pos % lcap
            else:
                page = b * pages + pos // 64
                at = ((page * HKV + g) * 64 + pos % 64) * HD + d
                av = ((page * HKV + g) * HD + d) * 64 + pos % 64
            cache[i, b] = [_cached(seed, i, which, x, dt).to(dt)
                           for which, x in ((0, at), (1, av))]
        return [x.double() for x in cache[i, b]]

    def attend(i, local, q, k, v):
        out = torch.empty_like(q)
        for b in range(B):
            ck, cv = cached(i, local, b)
            S = ck.shape[1]
            j, t = torch.arange(S + n, device=DEV), torch.arange(n, device=DEV)[:, None]
            mask = j <= S + t
            if local:
                mask = mask & (j > S + t - W)
            out[b] = _sdpa(q[b].contiguous(), torch.cat([ck, k[b]], 1), torch.cat([cv, v[b]], 1),
                           mask)
        return out

    a = _rms(net.t("tok_emb")[ids], net.t("anchor_norm"))[0]
    e = a * (1 + net.t("conv_w")[:, 0])
    h = net.pulses(e, range(ctx, ctx + n), attend, None, True)
    cap = CFG.logit_softcap
    return dict(logits=(cap * torch.tanh(net.head(h) / cap)).view(B * n, V))


def exact(case, seed):
    kind = case["kind"]
    if kind == "dense":
        return _exact_dense(case, seed)
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "prefill":
        return _exact_prefill(case, seed)
    if kind == "verify":
        return _exact_verify(case, seed)
    # generation: thousands of dependent passes, far over the time a check may take
    return None
