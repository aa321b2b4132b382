"""Performance cases of the RL step: what a training or rollout program has the library do.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges.
Sizes are those of ``summa_amd.configs`` (d_model 256 / 768 / 2048 decoders,
Q4G128 weights, GRPO groups of 8), of the published MoE layer (8192 tokens, d
512, expert width 768, 8 experts, top-2) and, where drawn, generic ones around
them. Every ``run`` is one pass through the public entry points (``ops``,
``model``, ``train``); ``exact`` restates its outputs in float64 torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from summa_amd import _lib, configs, ops, train
from summa_amd.model import Model, ModelConfig

DEV = "cuda"
GEOMETRY = {"d256": configs.CFG0_MODEL, "d768": configs.CFG1_MODEL, "d2048": configs.CFG2_MODEL}


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # The GRPO loss of one config[2] step (32 prompts x 8 rollouts x 512
        # tokens, rollouts that stopped early masked) with the host's one
        # validation readback: the smallest call, all latency.
        dict(name="grpo_loss", kind="grpo", groups=32, group=8, tokens=512, masked=True, kl=True),
        # Token log-probs and loss over bf16 logits of a 131072 vocabulary.
        dict(name="ce_rows", kind="ce", rows=8192, vocab=131072, logical=131072, dtype="bf16"),
        # A decoder layer's four 4-bit projections for a handful of requests:
        # serving, and the tail of a rollout.
        dict(name="q4_layer", kind="q4", m=8, geometry="d2048", x="f16"),
        # Attention of a training step, f32: forward with its log-sum-exp and
        # backward, one GRPO group of 8 x 1024 positions with 16 / 4 heads.
        dict(name="attention_train", kind="attn_train", batch=8, heads=16, kv_heads=4, seq=1024,
             head_dim=128, causal=True),
        # Attention of a prefill in bf16: 32 prompts of 512 tokens.
        dict(name="attention_prefill", kind="attn_prefill", batch=32, heads=16, kv_heads=4,
             seq=512, head_dim=128, causal=True, dtype="bf16"),
        # The fused linear head + cross-entropy of supervised training, loss
        # and all gradients, f32, d 768 and a 32768 vocabulary.
        dict(name="linear_ce", kind="linear_ce", tokens=4096, d=768, vocab=32768, logical=32768,
             bias=True),
        # Expert MLPs of a trained MoE layer, forward and backward, f32: 8192
        # tokens routed to the best 2 of 8 experts.
        dict(name="moe_mlp_train", kind="moe_train", tokens=8192, d=512, width=768, experts=8),
        # A whole MoE layer over 4-bit experts (router, route plan, both expert
        # projections, combine) at a recompute's token count.
        dict(name="moe_layer_q4", kind="moe_q4", tokens=8192, d=2048, width=1408, experts=32),
        # Greedy rollouts of the tiny fp32 decoder: launches and latency.
        dict(name="rollout_fp32", kind="rollout", geometry="d256", layers=2, quantized=False,
             prompts=4, group=8, prompt=32, new=32, temperature=0.0),
        # Sampled rollouts over 4-bit weights: 32 prompts x 8 rollouts, each
        # group's prompt shared; four of the decoder's equal layers.
        dict(name="rollout_q4", kind="rollout", geometry="d2048", layers=4, quantized=True,
             prompts=32, group=8, prompt=512, new=32, temperature=1.0),
        # The log-prob recompute of a 12-layer 4-bit decoder over 128 rollouts.
        dict(name="recompute_q4", kind="recompute", geometry="d768", layers=12, rows=128,
             prompt=128, new=256),
        # A policy update of one GRPO group: recompute with activations, loss,
        # backward and the optimizer step, bf16 matmul operands; two of the
        # decoder's equal layers beside its embedding and head.
        dict(name="policy_update", kind="policy", geometry="d2048", layers=2, group=8, prompt=512,
             new=512, planes=1),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grpo", "ce", "q4", "attn_train", "attn_prefill", "linear_ce", "moe_train",
                       "moe_q4", "rollout_fp32", "rollout_q4", "recompute", "policy"])
    if kind == "grpo":
        return dict(kind=kind, groups=_log(rng, 1, 64), group=rng.randint(2, 16),
                    tokens=_log(rng, 16, 1024), masked=rng.random() < 0.5, kl=rng.random() < 0.7)
    if kind == "ce":
        vocab = _log(rng, 4096, 131072)
        vocab = vocab if rng.random() < 0.3 else vocab // 128 * 128
        logical = vocab if rng.random() < 0.7 else vocab - rng.randint(1, 100)
        return dict(kind=kind, rows=_log(rng, 64, 8192), vocab=vocab, logical=logical,
                    dtype=rng.choice(["bf16", "f32"]))
    if kind == "q4":
        return dict(kind=kind, m=_log(rng, 1, 512), geometry=rng.choice(["d768", "d2048"]),
                    x=rng.choice(["f16", "bf16", "pair", "pair"]))
    if kind in ("attn_train", "attn_prefill"):
        kvh = rng.choice([2, 4, 8])
        c = dict(kind=kind, batch=rng.randint(1, 8), heads=kvh * rng.choice([1, 2, 4]),
                 kv_heads=kvh, seq=_log(rng, 32, 1024), head_dim=rng.choice([64, 128]),
                 causal=rng.random() < 0.8)
        if c["heads"] > 16:
            c["heads"] = 16
        if kind == "attn_prefill":
            c.update(batch=rng.randint(1, 32), dtype=rng.choice(["bf16", "f16"]))
        return c
    if kind == "linear_ce":
        vocab = _log(rng, 4096, 32768)
        vocab = vocab if rng.random() < 0.3 else vocab // 64 * 64
        return dict(kind=kind, tokens=_log(rng, 256, 4096), d=rng.choice([256, 384, 512, 768]),
                    vocab=vocab, logical=vocab - (rng.randint(1, 50) if rng.random() < 0.3 else 0),
                    bias=rng.random() < 0.5)
    if kind == "moe_train":
        return dict(kind=kind, tokens=_log(rng, 256, 8192), d=rng.choice([256, 512, 768, 1024]),
                    width=rng.choice([256, 512, 704, 768]), experts=rng.choice([4, 8, 16, 32]))
    if kind == "moe_q4":
        return dict(kind=kind, tokens=_log(rng, 32, 8192), d=rng.choice([512, 1024, 2048]),
                    width=rng.choice([512, 768, 1408]), experts=rng.choice([8, 16, 32]))
    if kind == "rollout_fp32":
        return dict(kind="rollout", geometry="d256", layers=rng.randint(1, 4), quantized=False,
                    prompts=rng.randint(2, 8), group=8, prompt=rng.randint(8, 64),
                    new=rng.randint(12, 32), temperature=rng.choice([0.0, 1.0]))
    if kind == "rollout_q4":
        big = rng.random() < 0.5
        return dict(kind="rollout", geometry="d2048" if big else "d768",
                    layers=rng.randint(1, 4) if big else rng.randint(2, 8), quantized=True,
                    prompts=rng.randint(16, 32), group=8, prompt=_log(rng, 32, 512),
                    new=rng.randint(8, 32), temperature=1.0)
    if kind == "recompute":
        big = rng.random() < 0.4
        return dict(kind=kind, geometry="d2048" if big else "d768",
                    layers=rng.randint(1, 3) if big else rng.randint(2, 12),
                    rows=_log(rng, 8, 64 if big else 128), prompt=_log(rng, 16, 128),
                    new=_log(rng, 16, 256))
    big = rng.random() < 0.4
    return dict(kind="policy", geometry="d2048" if big else "d768",
                layers=rng.randint(1, 2) if big else rng.randint(1, 6), group=rng.choice([4, 8]),
                prompt=_log(rng, 32, 256), new=_log(rng, 32, 256), planes=rng.choice([1, 3]))


# ----------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std).to(dtype)


def _ids(g, vocab, *shape):
    return torch.randint(0, vocab, shape, generator=g, device=DEV, dtype=torch.int32)


DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _model_cfg(case, max_seq, quantized):
    geo = dict(GEOMETRY[case["geometry"]])
    geo["layers"] = case["layers"]
    return ModelConfig(**geo, max_seq=max_seq, quantized=quantized)


def _weights(cfg, seed):
    """(name, layer, tensor) of a random decoder, N(0, 0.02) linears and unit
    norms; embedding values are bf16 numbers, as the 4-bit models store them."""
    g = _gen(seed)
    d, ffn, hd = cfg.d_model, cfg.ffn, cfg.head_dim
    ones = torch.ones(d, device=DEV)
    yield "embed", -1, _randn(g, cfg.vocab, d, std=0.02, dtype=torch.bfloat16).float()
    yield "lm_head", -1, _randn(g, cfg.vocab, d, std=0.02)
    yield "final_norm", -1, ones
    for layer in range(cfg.layers):
        yield "attn_norm", layer, ones
        yield "ffn_norm", layer, ones
        for name, n, k in (("qkv", (cfg.heads + 2 * cfg.kv_heads) * hd, d),
                           ("o", d, cfg.heads * hd), ("in", 2 * ffn, d), ("down", d, ffn)):
            yield name, layer, _randn(g, n, k, std=0.02)


def _build(cfg, seed):
    m = Model(cfg)
    for name, layer, w in _weights(cfg, seed):
        m.set_tensor(name, w, layer)
    return m


def _prompts(case, vocab, g):
    p = _ids(g, vocab, case["prompts"], case["prompt"])
    return p.repeat_interleave(case["group"], 0).contiguous()


def _route_counts(g, case):
    """Rows per expert of a top-2 router whose experts are unevenly liked."""
    E = case["experts"]
    logits = _randn(g, case["tokens"], E) + _randn(g, 1, E, std=0.5)
    return torch.bincount(logits.topk(2, 1).indices.reshape(-1), minlength=E).tolist()


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = dict(case=case)
    if kind == "grpo":
        shape = (case["groups"], case["group"], case["tokens"])
        cur = -_randn(g, *shape, std=2.0).abs() - 0.1
        s.update(rewards=torch.rand(shape[:2], generator=g, device=DEV), cur=cur,
                 beh=cur + _randn(g, *shape, std=0.1),
                 ref=cur + _randn(g, *shape, std=0.2) if case["kl"] else None, mask=None)
        if case["masked"]:  # rollouts end at their EOS
            n = torch.randint(1, shape[2] + 1, shape[:2], generator=g, device=DEV)
            at = torch.arange(shape[2], device=DEV)
            s["mask"] = (at < n[..., None]).float().contiguous()
    elif kind == "ce":
        rows, vocab = case["rows"], case["vocab"]
        x = torch.empty(rows, vocab, dtype=DTYPE[case["dtype"]], device=DEV)
        x.normal_(0.0, 3.0, generator=g)
        t = _ids(g, case["logical"], rows)
        x[torch.arange(rows, device=DEV), t.long()] += 8.0
        s.update(x=x, t=t)
    elif kind == "q4":
        geo = GEOMETRY[case["geometry"]]
        d, ffn, hd = geo["d_model"], geo["ffn"], geo["head_dim"]
        shapes = dict(qkv=((geo["heads"] + 2 * geo["kv_heads"]) * hd, d),
                      o=(d, geo["heads"] * hd), up=(2 * ffn, d), down=(d, ffn))
        s["w"] = {k: ops.Q4Weight.quantize(_randn(g, *sh, std=0.02)) for k, sh in shapes.items()}
        x = {k: _randn(g, case["m"], shapes[k][1]) for k in ("qkv", "o", "up")}
        pair = case["x"] == "pair"
        s["x"] = {k: ops.f16_pair(v) if pair else v.to(DTYPE[case["x"]]) for k, v in x.items()}
        s["epi"] = {"f16": _lib.SM_EPI_SWIGLU_F16, "bf16": _lib.SM_EPI_SWIGLU_BF16,
                    "pair": _lib.SM_EPI_SWIGLU_F16X2}[case["x"]]
        s["ws"] = {k: ops.q4_workspace(case["m"], *sh, s["epi"] if k == "up" else
                                       _lib.SM_EPI_STORE_F32, DEV) for k, sh in shapes.items()}
    elif kind in ("attn_train", "attn_prefill"):
        B, H, KVH, S, hd = (case[k] for k in ("batch", "heads", "kv_heads", "seq", "head_dim"))
        dt = DTYPE[case.get("dtype", "f32")]
        s.update(q=_randn(g, B, H, S, hd, dtype=dt), k=_randn(g, B, KVH, S, hd, dtype=dt),
                 v=_randn(g, B, KVH, S, hd, dtype=dt))
        if kind == "attn_train":
            s["do"] = _randn(g, B, H, S, hd)
    elif kind == "linear_ce":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        s.update(h=_randn(g, T, d), w=_randn(g, V, d, std=0.02),
                 b=_randn(g, V, std=0.02) if case["bias"] else None,
                 t=_ids(g, case["logical"], T), go=torch.ones(1, device=DEV))
    elif kind == "moe_train":
        d, width, E = case["d"], case["width"], case["experts"]
        s.update(counts=_route_counts(g, case), x=_randn(g, 2 * case["tokens"], d),
                 wi=_randn(g, E, d, 2 * width, std=0.02), wd=_randn(g, E, width, d, std=0.02),
                 grad=_randn(g, 2 * case["tokens"], d))
    elif kind == "moe_q4":
        d, width, E = case["d"], case["width"], case["experts"]
        s.update(h=ops.f16_pair(_randn(g, case["tokens"], d)),
                 router=_randn(g, E, d, std=1 / math.sqrt(d)),
                 up=ops.ExpertBank.quantize(_randn(g, E, 2 * width, d, std=0.02)),
                 down=ops.ExpertBank.quantize(_randn(g, E, d, width, std=0.02)))
    elif kind == "rollout":
        cfg = _model_cfg(case, case["prompt"] + case["new"], case["quantized"])
        m = _build(cfg, seed)
        m.set_prompt_groups(case["group"])
        m.bind_workspace(case["prompts"] * case["group"], case["prompt"], case["new"])
        s.update(model=m, prompts=_prompts(case, cfg.vocab, g), seed=int(seed))
    elif kind == "recompute":
        cfg = _model_cfg(case, case["prompt"] + case["new"], True)
        m = _build(cfg, seed)
        m.bind_workspace(case["rows"], case["prompt"], case["new"])
        s.update(model=m, prompts=_ids(g, cfg.vocab, case["rows"], case["prompt"]),
                 tokens=_ids(g, cfg.vocab, case["rows"], case["new"]))
    elif kind == "policy":
        cfg = _model_cfg(case, case["prompt"] + case["new"], True)
        w = {}
        for name, layer, t in _weights(cfg, seed):
            w.setdefault(name, []).append(t)
        w = {k: torch.stack(v) if k in train.LAYER_KEYS else v[0] for k, v in w.items()}
        n, N = case["group"], case["new"]
        lp = _randn(g, n, N, std=0.1) - (math.log(cfg.vocab) + 0.4)
        s.update(cfg=cfg, policy=train.Policy(cfg, w, DEV, matmul_planes=case["planes"]),
                 prompts=_ids(g, cfg.vocab, 1, case["prompt"]).expand(n, -1).contiguous(),
                 tokens=_ids(g, cfg.vocab, n, N), beh=lp, ref=lp + _randn(g, n, N, std=0.05),
                 rewards=torch.rand((1, n), generator=g, device=DEV))
    return s


# ------------------------------------------------------------------- runs --

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "grpo":
        return ops.grpo_loss_batched(s["rewards"], s["cur"], s["beh"], s["ref"], s["mask"],
                                     kl_coefficient=0.04 if case["kl"] else 0.0)
    if kind == "ce":
        return ops.ce_rows(s["x"], s["t"], case["logical"], want_lse=True)
    if kind == "q4":
        w, x, ws, pair = s["w"], s["x"], s["ws"], case["x"] == "pair"
        qkv = ops.q4_matmul(w["qkv"], x["qkv"], pair=pair, workspace=ws["qkv"])
        o = ops.q4_matmul(w["o"], x["o"], pair=pair, workspace=ws["o"])
        u = ops.q4_matmul(w["up"], x["up"], epilogue=s["epi"], pair=pair, workspace=ws["up"])
        return qkv, o, ops.q4_matmul(w["down"], u, pair=pair, workspace=ws["down"])
    if kind == "attn_train":
        q, k, v, causal = s["q"], s["k"], s["v"], case["causal"]
        out, lse = ops.attention(q, k, v, causal, want_lse=True)
        return (out, lse) + ops.attention_backward(q, k, v, out, s["do"], lse, causal)
    if kind == "attn_prefill":
        return ops.attention(s["q"], s["k"], s["v"], case["causal"])
    if kind == "linear_ce":
        a = (s["h"], s["w"], s["b"], s["t"])
        loss = ops.linear_cross_entropy(*a, logical_vocab=case["logical"])
        return (loss,) + ops.linear_cross_entropy_backward(*a, s["go"],
                                                           logical_vocab=case["logical"])
    if kind == "moe_train":
        x, wi, wd, counts, width = s["x"], s["wi"], s["wd"], s["counts"], case["width"]
        out, proj, hid = ops.grouped_swiglu_mlp(x, wi, wd, counts, width)
        return (out,) + ops.grouped_swiglu_mlp_backward(x, wi, wd, counts, proj, hid, s["grad"],
                                                        width)
    if kind == "moe_q4":
        idx, w, _ = ops.moe_top2_indices(s["h"], s["router"], pair=True)
        plan = ops.moe_route_plan(idx, case["experts"])
        u = ops.grouped_q4_matmul(s["up"], s["h"], plan, gather=True,
                                  epilogue=_lib.SM_EPI_SWIGLU_F16X2, pair=True)
        routed = ops.grouped_q4_matmul(s["down"], u, plan, gather=False, pair=True)
        x = torch.zeros(case["tokens"], case["d"], device=DEV)
        return idx, w, ops.moe_route_combine(routed, w, plan, x)
    if kind == "rollout":
        return s["model"].generate(s["prompts"], case["new"], temperature=case["temperature"],
                                   seed=s["seed"])
    if kind == "recompute":
        return s["model"].logprobs(s["prompts"], s["tokens"])
    pol = s["policy"]
    out = pol.prepare(None, s["prompts"], s["tokens"], s["beh"], s["rewards"],
                      reference_lp=s["ref"])
    grads = {name: pol.tensor(name, gradient=True) for name in ("embed", "lm_head", "final_norm")}
    for layer in range(case["layers"]):
        for name in train.LAYER_KEYS:
            grads[f"{name}{layer}"] = pol.tensor(name, layer, gradient=True)
    return dict(lp=out["lp_cur"], stats=out["stats"], dlp=out["dlp"], grads=grads,
                norm=pol.optimizer_step())


# ------------------------------------------------------------------- work --

def _layer_params(geo):
    d, hd = geo["d_model"], geo["head_dim"]
    return (geo["heads"] * 2 + geo["kv_heads"] * 2) * hd * d + 3 * geo["ffn"] * d


def _attn_flops(batch, heads, seq, hd, causal):
    return 4 * batch * heads * hd * (seq * (seq + 1) / 2 if causal else seq * seq)


def work(case):
    kind = case["kind"]
    if kind == "grpo":
        n = case["groups"] * case["group"] * case["tokens"]
        return dict(bytes=4 * n * (3 + case["masked"] + case["kl"]), flops=40 * n)
    if kind == "ce":
        e = 2 if case["dtype"] == "bf16" else 4
        return dict(bytes=case["rows"] * case["logical"] * e + 12 * case["rows"],
                    flops=4 * case["rows"] * case["logical"])
    if kind == "q4":
        geo, m = GEOMETRY[case["geometry"]], case["m"]
        d, hd, ffn = geo["d_model"], geo["head_dim"], geo["ffn"]
        qn, e = (geo["heads"] + 2 * geo["kv_heads"]) * hd, 4 if case["x"] == "pair" else 2
        n = _layer_params(geo)
        act = m * (2 * d + geo["heads"] * hd) * e + m * 4 * (qn + 2 * d) + 2 * m * ffn * e
        return dict(bytes=n * (0.5 + 2 / 128) + act, flops=2 * m * n)
    if kind in ("attn_train", "attn_prefill"):
        B, H, KVH, S, hd = (case[k] for k in ("batch", "heads", "kv_heads", "seq", "head_dim"))
        f = _attn_flops(B, H, S, hd, case["causal"])
        if kind == "attn_prefill":
            return dict(bytes=2 * B * S * hd * (2 * H + 2 * KVH), flops=f)
        return dict(bytes=4 * B * S * hd * (2 * (2 * H + 2 * KVH) + 2 * H + 2 * KVH),
                    flops=3.5 * f)
    if kind == "linear_ce":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        return dict(bytes=4 * (3 * T * d + 3 * V * d), flops=6.0 * T * d * V)
    if kind == "moe_train":
        R, d, w, E = 2 * case["tokens"], case["d"], case["width"], case["experts"]
        return dict(bytes=4 * (4 * R * d + 4 * R * 3 * w + 3 * E * 3 * d * w),
                    flops=3 * 2.0 * R * 3 * d * w)
    if kind == "moe_q4":
        T, d, w, E = case["tokens"], case["d"], case["width"], case["experts"]
        used = min(E, 2 * T)
        return dict(bytes=used * 3 * w * d * (0.5 + 2 / 128) + T * d * 8 + 2 * T * (w + d) * 4,
                    flops=2 * 2.0 * T * 3 * w * d + 2.0 * T * d * E)
    geo = GEOMETRY[case["geometry"]]
    d, hd, H, KVH, V = (geo[k] for k in ("d_model", "head_dim", "heads", "kv_heads", "vocab"))
    Ly, P, N = case["layers"], case["prompt"], case["new"]
    n = Ly * _layer_params(geo)
    if kind == "rollout":
        S, groups = case["prompts"] * case["group"], case["prompts"]
        wb, kvb = (0.5 + 2 / 128, 2) if case["quantized"] else (4, 4)
        kv = 2 * KVH * hd * kvb * Ly
        own = S * N * (N - 1) / 2
        by = N * (n + V * d) * wb + kv * (groups * P * N + own) + 4 * S * V * N
        fl = 2.0 * (n * (groups * P + S * (N - 1)) + V * d * S * N)
        fl += Ly * (_attn_flops(groups, H, P, hd, True) + 4 * H * hd * (S * P * N + own))
        return dict(bytes=by, flops=fl)
    if kind == "recompute":
        S, L = case["rows"], P + N - 1
        return dict(bytes=(n + V * d) * (0.5 + 2 / 128) + 4 * S * N,
                    flops=2.0 * (n * S * L + V * d * S * N) +
                    Ly * _attn_flops(S, H, L, hd, True))
    S, L = case["group"], P + N - 1
    params = n + 2 * V * d
    return dict(bytes=params * (4 + 4 + 3 * 8),
                flops=6.0 * (n * S * L + V * d * S * N) +
                3.5 * Ly * _attn_flops(S, H, L, hd, True))


def tolerance(case):
    """About four times the distance to ``exact`` that was measured."""
    kind = case["kind"]
    if kind == "grpo":  # f64 sums, f32 results: 3e-8
        return dict(rel=2e-7)
    if kind == "ce":  # f32 sums over a row: 7e-8
        return dict(rel=1e-6)
    if kind == "q4":  # f32 sums; the SwiGLU output is rounded to x's type between
        return dict(rel={"pair": 2e-6, "f16": 8e-4, "bf16": 7e-3}[case["x"]])
    if kind == "attn_prefill":  # the output type's rounding
        return dict(rel={"f16": 1e-3, "bf16": 7e-3}[case["dtype"]])
    if kind in ("attn_train", "moe_train", "linear_ce"):  # f32 sums: up to 1.3e-6, 1e-6, 2.3e-6
        return dict(rel=1e-5 if kind == "linear_ce" else 5e-6)
    if kind == "moe_q4":  # f32 sums, 7e-7; no pair of experts is expected to change
        return dict(rel=4e-6, differ=1e-4)
    if kind == "rollout":
        # A token whose two best candidates are closer than the rounding may go
        # either way, and its rollout goes on differently from there. f32 logits
        # move by 1e-6 and hardly ever meet one; 4-bit models (16-bit keys and
        # values) by 1e-4, about once in 10000 tokens.
        if not case["quantized"]:
            return dict(rel=1e-5, differ=1e-2)
        return dict(rel=2e-2, max=0.99, differ=1e-2)
    if kind == "recompute":  # 16-bit keys and values: 2.4e-5
        return dict(rel=1e-4)
    # bf16 operands throughout: 3e-2 to exact, dominated by exp(lp - behaviour);
    # three planes: f32 sums, 4e-6
    return dict(rel=3e-2, max=0.99) if case["planes"] == 1 else dict(rel=2e-5)


# ------------------------------------------------------------------ exact --

def _dequantize(w):
    """Q4G128 round trip of dense [N, K] weights, in f64."""
    return _codes(ops.Q4Weight.quantize(w))


def _codes(w):
    """f64 values of a Q4Weight from its row-major codes (two's complement, the
    even element in the low half of a byte) and bf16 scales per 128 values."""
    c = w.codes.to(torch.int32)
    q = torch.stack([c & 15, c >> 4], 1).reshape(-1, 128)
    q = torch.where(q > 7, q - 16, q).double()
    s = (w.scales.to(torch.int32) << 16).view(torch.float32).double()
    return (q * s[:, None]).reshape(w.n, w.k)


def _f64(x, pair):
    if not pair:
        return x.double()
    k = x.shape[1] // 2
    return x[:, :k].double() + x[:, k:].double()


def _attention(q, k, v, causal):
    """[H, S, hd] f64 queries over [KVH, S, hd]: (out, log-sum-exp)."""
    rep = q.shape[0] // k.shape[0]
    sc = q @ k.repeat_interleave(rep, 0).transpose(1, 2) / math.sqrt(q.shape[-1])
    if causal:
        n = sc.shape[-1]
        sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool, device=sc.device).triu(1),
                            float("-inf"))
    return torch.softmax(sc, -1) @ v.repeat_interleave(rep, 0), torch.logsumexp(sc, -1)


def _swiglu(u):
    half = u.shape[-1] // 2
    return F.silu(u[..., :half]) * u[..., half:]


def _decoder_lp(w, cfg, prompts, tokens):
    """Log-probs [S, N] of tokens after prompts under the decoder w, in f64."""
    S, P = prompts.shape
    N = tokens.shape[1]
    L, H, KVH, hd = P + N - 1, cfg.heads, cfg.kv_heads, cfg.head_dim
    ids = torch.cat([prompts, tokens[:, :N - 1]], 1).long()

    def rms(x, gain):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg.norm_eps) * gain

    freq = float(cfg.rope_theta) ** (-2.0 * np.arange(hd // 2) / hd)
    ang = np.arange(L)[:, None] * freq[None, :]
    tab = torch.from_numpy(np.stack([np.cos(ang), np.sin(ang)], -1).astype(np.float32))
    tab = tab.to(DEV).double()
    cos, sin = tab[:, None, :, 0], tab[:, None, :, 1]

    def rope(x):  # [S, L, heads, hd], adjacent pairs
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)

    x = w["embed"][ids]
    for i in range(cfg.layers):
        qkv = rms(x, w["attn_norm"][i]) @ w["qkv"][i].T
        q = rope(qkv[..., :H * hd].reshape(S, L, H, hd)).transpose(1, 2)
        k = rope(qkv[..., H * hd:(H + KVH) * hd].reshape(S, L, KVH, hd)).transpose(1, 2)
        v = qkv[..., (H + KVH) * hd:].reshape(S, L, KVH, hd).transpose(1, 2)
        o = torch.stack([_attention(q[r], k[r], v[r], True)[0] for r in range(S)])
        x = x + o.transpose(1, 2).reshape(S, L, H * hd) @ w["o"][i].T
        x = x + _swiglu(rms(x, w["ffn_norm"][i]) @ w["in"][i].T) @ w["down"][i].T
    hf = rms(x, w["final_norm"])[:, P - 1:P - 1 + N]
    lp = torch.log_softmax(hf @ w["lm_head"].T, -1)
    return lp.gather(-1, tokens.long()[..., None])[..., 0]


def _decoder_weights(cfg, seed):
    """The f64 decoder that a 4-bit model of these weights stands for."""
    w = {}
    for name, _, t in _weights(cfg, seed):
        v = _dequantize(t) if name in ("qkv", "o", "in", "down", "lm_head") else t.double()
        w.setdefault(name, []).append(v)
    return {k: v if k in train.LAYER_KEYS else v[0] for k, v in w.items()}


def _grpo(rewards, cur, beh, ref, mask, eps=0.2, beta=0.04):
    """The clipped policy-gradient + k3 KL loss per group, in f64."""
    r = rewards.double()
    mean, std = r.mean(1, keepdim=True), r.std(1, unbiased=False, keepdim=True)
    adv = (r - mean) / std.clamp_min(1e-6)
    mk = torch.ones_like(cur) if mask is None else mask.double()
    ts = mk / (r.shape[1] * mk.sum(-1, keepdim=True))
    rho, a = torch.exp(cur - beh), adv[..., None]
    clip = rho.clamp(1 - eps, 1 + eps)
    surr = torch.minimum(rho * a, clip * a)
    kl = torch.exp(ref - cur) - (ref - cur) - 1 if ref is not None else torch.zeros_like(cur)
    loss = -(ts * (surr - beta * kl)).sum((1, 2))
    clipped = ((surr == clip * a) & (rho != clip) & (mk != 0)).double().sum((1, 2))
    stats = torch.stack([loss, mean[:, 0], std[:, 0], (ts * kl).sum((1, 2)),
                         clipped / mk.sum((1, 2))], 1)
    return stats, adv, loss


def exact(case, seed):
    kind = case["kind"]
    if kind == "rollout":
        return None  # sampled tokens
    if kind == "recompute":
        cfg = _model_cfg(case, case["prompt"] + case["new"], True)
        g = _gen(seed)
        prompts = _ids(g, cfg.vocab, case["rows"], case["prompt"])
        tokens = _ids(g, cfg.vocab, case["rows"], case["new"])
        w = _decoder_weights(cfg, seed)
        return torch.cat([_decoder_lp(w, cfg, prompts[r:r + 4], tokens[r:r + 4])
                          for r in range(0, case["rows"], 4)])
    s = prepare(case, seed)
    if kind == "grpo":
        cur = s["cur"].double().requires_grad_(True)
        ref = None if s["ref"] is None else s["ref"].double()
        stats, adv, loss = _grpo(s["rewards"], cur, s["beh"].double(), ref, s["mask"])
        loss.sum().backward()
        return dict(stats=stats.detach(), advantages=adv, dlp=cur.grad, flags=None)
    if kind == "ce":
        lp, lse = [], []
        for r in range(0, case["rows"], 512):
            x = s["x"][r:r + 512, :case["logical"]].double()
            lse.append(torch.logsumexp(x, 1))
            lp.append(x.gather(1, s["t"][r:r + 512].long()[:, None])[:, 0] - lse[-1])
        lp, lse = torch.cat(lp), torch.cat(lse)
        return lp, -lp.mean().reshape(1), lse
    if kind == "q4":
        pair = case["x"] == "pair"
        x = {k: _f64(v, pair) for k, v in s["x"].items()}
        w = {k: _codes(v) for k, v in s["w"].items()}
        u = _swiglu(x["up"] @ w["up"].T)
        return x["qkv"] @ w["qkv"].T, x["o"] @ w["o"].T, u @ w["down"].T
    if kind in ("attn_train", "attn_prefill"):
        got = []
        for b in range(case["batch"]):
            q, k, v = (s[n][b].double().requires_grad_(kind == "attn_train") for n in "qkv")
            out, lse = _attention(q, k, v, case["causal"])
            if kind == "attn_train":
                out.backward(s["do"][b].double())
                got.append((out.detach(), lse.detach(), q.grad, k.grad, v.grad))
            else:
                got.append((out,))
        got = [torch.stack(t) for t in zip(*got)]
        if kind == "attn_prefill":
            return got[0]
        got[1] = got[1].reshape(-1, case["seq"])
        return tuple(got)
    if kind == "linear_ce":
        h, w = (s[n].double().requires_grad_(True) for n in "hw")
        b = s["b"].double().requires_grad_(True) if case["bias"] else None
        logits = F.linear(h, w, b)[:, :case["logical"]]
        loss = F.cross_entropy(logits, s["t"].long())
        loss.backward()
        return loss.detach().reshape(1), h.grad, w.grad, b.grad if case["bias"] else None
    if kind == "moe_train":
        x, wi, wd = (s[n].double().requires_grad_(True) for n in ("x", "wi", "wd"))
        out = torch.cat([_swiglu(rows @ wi[e]) @ wd[e]
                         for e, rows in enumerate(x.split(s["counts"]))])
        out.backward(s["grad"].double())
        return out.detach(), x.grad, wi.grad, wd.grad
    if kind == "moe_q4":
        h, E = _f64(s["h"], True), case["experts"]
        top, idx = (h @ s["router"].double().T).topk(2, 1)
        pw = torch.softmax(top, 1)
        # the same draws as prepare's, dequantized here
        g = _gen(seed)
        _randn(g, case["tokens"], case["d"])
        _randn(g, E, case["d"])
        up = _randn(g, E, 2 * case["width"], case["d"], std=0.02)
        down = _randn(g, E, case["d"], case["width"], std=0.02)
        out = torch.zeros_like(h)
        for e in range(E):
            t, j = torch.where(idx == e)
            y = _swiglu(h[t] @ _dequantize(up[e]).T) @ _dequantize(down[e]).T
            out.index_add_(0, t, y * pw[t, j][:, None])
        return None, pw, out
    w = _decoder_weights(s["cfg"], seed)
    leaves = [t for v in w.values() for t in (v if isinstance(v, list) else [v])]
    for t in leaves:
        t.requires_grad_(True)
    lp = _decoder_lp(w, s["cfg"], s["prompts"], s["tokens"])
    at = lp.detach()[None].requires_grad_(True)
    stats, _, loss = _grpo(s["rewards"], at, s["beh"][None].double(), s["ref"][None].double(),
                           None)
    loss.sum().backward()
    lp.backward(at.grad[0])
    grads = {name: w[name].grad for name in ("embed", "lm_head", "final_norm")}
    grads.update({f"{name}{i}": w[name][i].grad for name in train.LAYER_KEYS
                  for i in range(case["layers"])})
    norm = math.sqrt(sum(float(t.grad.square().sum()) for t in leaves))
    return dict(lp=lp.detach(), stats=stats.detach(), dlp=at.grad[0], grads=grads, norm=norm)
