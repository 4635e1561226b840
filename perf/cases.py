"""Performance cases of the speculative rollout: what a rollout program calls, over the sizes of this
repository's model configurations.

A case is one call (or the few calls that belong together) of the public entry points: a draw from
logits, tree attention, the tree-verify forward, prefill, the Medusa and chain proposals, the lazy
acceptance walk with its KV compaction, and a whole small rollout. ``listed()`` holds the sizes that
are followed over time, ``draw(rng)`` gives others of the same ranges.
"""
from __future__ import annotations

import dataclasses
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ss-grpo_amd"))

from flashgrpo_amd import kernels as K  # noqa: E402
from flashgrpo_amd.decoding import FlashMedusaConfig, FlashMedusaDecoder  # noqa: E402
from flashgrpo_amd.models import MedusaHeads, TargetConfig, TargetModel  # noqa: E402
from flashgrpo_amd.models.target import KVCache  # noqa: E402

DEV = "cuda"
MODELS = {"tiny": TargetConfig.tiny, "1.5b": TargetConfig.qwen25_1p5b, "7b": TargetConfig.qwen25_7b,
          "8b": TargetConfig.llama31_8b, "14b": TargetConfig.qwen25_14b}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The root draw of a small fp32 rollout: the shortest call there is, latency alone.
        dict(name="draw-small", kind="draw", rows=8, vocab=32000, dtype="fp32", temperature=1.0, top_p=1.0, top_k=0),
        # The root draw of a 64-sequence rollout with the sampling default, nucleus 0.95.
        dict(name="draw-top-p", kind="draw", rows=64, vocab=152064, dtype="bf16", temperature=1.0, top_p=0.95, top_k=0),
        # The same draw with a top-k cut and a temperature, the other restricted option.
        dict(name="draw-top-k", kind="draw", rows=32, vocab=151936, dtype="bf16", temperature=0.7, top_p=1.0, top_k=50),
        # One layer's tree attention of a verify round: the kernel that reads the KV cache.
        dict(name="attention-verify-7b", kind="attention", model="7b", batch=64, prefix=2048, nodes=29, causal=False),
        # One layer's attention of a prefill chunk whose rows already hold a ragged prefix.
        dict(name="attention-chunk-8b", kind="attention", model="8b", batch=4, prefix=1000, nodes=1024, causal=True),
        # The tree-verify forward of a small batch (launch- and latency-bound layers).
        dict(name="verify-1.5b", kind="verify", model="1.5b", layers=2, batch=32, prefix=512, nodes=13),
        # One decoder layer of the large verify forward (matrix products of 1,856 rows).
        dict(name="verify-7b", kind="verify", model="7b", layers=1, batch=64, prefix=2048, nodes=29),
        # Prompts of unequal length before a rollout.
        dict(name="prefill-8b", kind="prefill", model="8b", layers=1, batch=4, prompt=777),
        # Medusa heads, tied LM head and per-row candidates: what opens a round.
        dict(name="proposals-7b", kind="proposals", model="7b", batch=64, heads=4, kmax=4),
        # One depth of chain proposals: LM head and candidates of every parent state, then the children's states.
        dict(name="chain-8b", kind="chain", model="8b", batch=96, parents=4, kmax=2),
        # The lazy acceptance walk: LM-head rows of the current nodes, a draw per step, clamp, KV compaction.
        dict(name="walk-7b", kind="walk", model="7b", layers=28, batch=64, prefix=512, tree="4,2,1,1"),
        # A whole rollout of a small fp32 model: prefill and 12 verify rounds with everything between them.
        dict(name="rollout-tiny", kind="rollout", model="tiny", prompts=4, repeats=2, prefix=256, rounds=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _one(rng):
    kind = rng.choice(["draw", "draw", "attention", "attention", "verify", "verify", "prefill", "proposals", "chain",
                       "walk", "rollout"])
    model = rng.choice(["1.5b", "7b", "8b", "14b"])
    if kind == "draw":
        mode = rng.choice(["plain", "top_p", "top_k", "both"])
        return dict(kind=kind, rows=_log(rng, 1, 128), vocab=_log(rng, 30000, 152064), dtype=rng.choice(["bf16", "bf16", "fp32"]),
                    temperature=rng.choice([1.0, 0.7, 0.6]), top_p=rng.choice([0.95, 0.9]) if mode in ("top_p", "both") else 1.0,
                    top_k=rng.choice([20, 50, 200]) if mode in ("top_k", "both") else 0)
    if kind == "attention":
        causal = rng.random() < 0.4
        return dict(kind=kind, model=rng.choice([model, model, "tiny"]), batch=_log(rng, 1, 8 if causal else 96), prefix=_log(rng, 64, 4096),
                    nodes=_log(rng, 65, 1024) if causal else rng.randint(2, 64), causal=causal)
    if kind == "verify":
        return dict(kind=kind, model=rng.choice([model, model, "tiny"]), layers=rng.randint(1, 2), batch=_log(rng, 1, 96), prefix=_log(rng, 64, 2048),
                    nodes=rng.randint(5, 48))
    if kind == "prefill":
        return dict(kind=kind, model=rng.choice([model, model, "tiny"]), layers=rng.randint(1, 2), batch=_log(rng, 1, 8), prompt=_log(rng, 32, 1500))
    if kind == "proposals":
        return dict(kind=kind, model=model, batch=_log(rng, 1, 128), heads=rng.randint(3, 4), kmax=rng.randint(2, 5))
    if kind == "chain":
        return dict(kind=kind, model=model, batch=_log(rng, 1, 96), parents=rng.choice([1, 1, 2, 4]), kmax=rng.randint(1, 4))
    if kind == "walk":
        return dict(kind=kind, model=model, layers=rng.choice([8, 28]), batch=_log(rng, 1, 96), prefix=_log(rng, 64, 512),
                    tree=rng.choice(["4,2,1,1", "4,2", "3,2,1", "4,2,1"]))
    return dict(kind=kind, model="tiny", prompts=rng.randint(1, 4), repeats=rng.randint(1, 4), prefix=_log(rng, 32, 256),
                rounds=rng.randint(3, 12))


def draw(rng):
    """One more case of the listed ones' ranges, none dearer than the dearest of them."""
    top = max(_cost(c) for c in listed())
    while True:
        c = _one(rng)
        if _cost(c) <= top:
            return c


def _cost(case):
    w = work(case)
    return w["bytes"] + w["flops"] / 300


# ------------------------------------------------------------------ sizes
def _cfg(case):
    return dataclasses.replace(MODELS[case["model"]](), num_layers=int(case.get("layers", 0)))


def _dtype(case):
    return torch.float32 if case.get("model") == "tiny" or case.get("dtype") == "fp32" else torch.bfloat16


def _layer_params(cfg):
    return cfg.hidden * ((2 * cfg.q_heads + 2 * cfg.kv_heads) * cfg.head_dim + 3 * cfg.intermediate)


def work(case):
    kind = case["kind"]
    e = 4 if _dtype(case) == torch.float32 else 2
    if kind == "draw":
        return dict(bytes=case["rows"] * case["vocab"] * e + case["rows"] * 4, flops=0)
    cfg = _cfg(case)
    H, V, d, Hq, Hkv = cfg.hidden, cfg.vocab, cfg.head_dim, cfg.q_heads, cfg.kv_heads
    B = case.get("batch", 0)

    def attention(n, prefix, causal):
        keys = B * (prefix * 7 // 8 + n)   # ragged prefixes: 7/8 of the longest on average
        pairs = B * n * (prefix * 7 // 8 + (n // 2 if causal else n))
        return 2 * Hkv * keys * d * e + 2 * B * n * Hq * d * e, 4 * Hq * d * pairs

    if kind == "attention":
        b, f = attention(case["nodes"], case["prefix"], case["causal"])
        return dict(bytes=b, flops=f)
    if kind in ("verify", "prefill"):
        n, prefix = (case["nodes"], case["prefix"]) if kind == "verify" else (case["prompt"], 0)
        b, f = attention(n, prefix, kind == "prefill")
        rows, P = B * n, _layer_params(cfg)
        return dict(bytes=cfg.num_layers * (P * e + b) + 2 * rows * H * e, flops=cfg.num_layers * (2 * rows * P + f))
    if kind == "proposals":
        R = B * case["heads"]
        return dict(bytes=(case["heads"] * H * H + V * H) * e + B * H * e + R * case["kmax"] * 8,
                    flops=2 * R * H * (H + V))
    if kind == "chain":
        R, C = B * case["parents"], B * case["parents"] * case["kmax"]
        return dict(bytes=V * H * e + R * H * 4 + C * H * (8 + e) + 3 * H * (H // 8) * 4, flops=2 * R * H * V + 6 * C * H * (H // 8))
    if kind == "walk":
        D = len(case["tree"].split(","))
        return dict(bytes=D * (V * H * e + B * (H + V) * e), flops=2 * D * B * H * V)
    rows = case["prompts"] * case["repeats"]
    per = 4 * (_layer_params(cfg)) + V * H
    return dict(bytes=case["rounds"] * per * e * 2, flops=2 * per * (case["rounds"] * rows * 13 + case["prompts"] * case["prefix"]))


# ------------------------------------------------------------------ inputs
def _gen(seed, *more):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + sum((i + 1) * 7919 * int(m) for i, m in enumerate(more))) % (1 << 62))


def _normal(g, shape, dtype, std):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _lengths(batch, prefix, seed):
    """Ragged committed lengths: between three quarters of the longest and the longest."""
    r = random.Random(int(seed) + 1)
    return [prefix - r.randint(0, prefix // 4) for _ in range(batch)]


def _tree(nodes, seed):
    """(parents, depths, ancestor-or-self bits) of a random tree in breadth-first order."""
    r = random.Random(int(seed) * 31 + nodes)
    par, dep = [-1], [0]
    for n in range(1, nodes):
        p = max(par[-1], r.randint(max(0, (n - 1) // 4 - 1), (n - 1) // 2)) if n > 1 else 0
        par.append(min(p, n - 1))
        dep.append(dep[par[-1]] + 1)
    bits = []
    for n in range(nodes):
        bits.append((bits[par[n]] if n else 0) | (1 << n))
    return par, dep, bits


def _masks(bits):
    return torch.from_numpy(np.array(bits, dtype=np.uint64).view(np.int64)).to(DEV)


def _weights(cfg, dtype, seed):
    """Random weights of the scale that trained models start from (std 0.02; norms near 1)."""
    g = _gen(seed, 3)
    H, d, I = cfg.hidden, cfg.head_dim, cfg.intermediate
    W = (cfg.q_heads + 2 * cfg.kv_heads) * d
    w = {"embed": _normal(g, (cfg.vocab, H), dtype, 0.02), "final_norm": 1 + _normal(g, (H,), dtype, 0.1), "layers": []}
    for _ in range(cfg.num_layers):
        w["layers"].append({
            "input_norm": 1 + _normal(g, (H,), dtype, 0.1), "qkv_w": _normal(g, (W, H), dtype, 0.02),
            "qkv_b": _normal(g, (W,), dtype, 0.1) if cfg.qkv_bias else None,
            "o_w": _normal(g, (H, cfg.q_heads * d), dtype, 0.02), "post_norm": 1 + _normal(g, (H,), dtype, 0.1),
            "gate_up_w": _normal(g, (2 * I, H), dtype, 0.02), "down_w": _normal(g, (H, I), dtype, 0.02)})
    w["lm_head"] = w["embed"] if cfg.tie_word_embeddings else _normal(g, (cfg.vocab, H), dtype, 0.02)
    return w


def _heads(cfg, n, seed):
    """Medusa heads as the trainer holds them: fp32 masters on the device."""
    g = _gen(seed, 5)
    m = MedusaHeads(cfg.hidden, cfg.vocab, n).to(DEV)
    with torch.no_grad():
        for hd in m.heads:
            hd.fc.weight.normal_(0.0, 0.02, generator=g)
            hd.fc.bias.normal_(0.0, 0.02, generator=g)
        c = m.chain_cell
        for p in (c.state_proj.weight, c.token_proj.weight, c.out_proj.weight, c.out_proj.bias):
            p.normal_(0.0, 0.02, generator=g)
    return m.requires_grad_(False)


def _logits(rows, vocab, dtype, seed):
    """Rows as an LM head gives them: a broad bulk and a few tokens that stand out."""
    g = _gen(seed, 1)
    x = torch.empty(rows, vocab, dtype=torch.float32, device=DEV).normal_(0.0, 2.0, generator=g)
    at = torch.randint(0, vocab, (rows, 24), device=DEV, generator=g)
    up = 6.0 + 8.0 * torch.rand(rows, 24, device=DEV, generator=g)
    return x.scatter_add_(1, at, up).to(dtype)


def _attention_inputs(case, seed):
    cfg, dt, B, N, P = _cfg(case), _dtype(case), case["batch"], case["nodes"], case["prefix"]
    g = _gen(seed, 2)
    cap = P + N + 80
    kv = _normal(g, (2, B, cfg.kv_heads, cap, cfg.head_dim), dt, 1.0)
    lens = _lengths(B, P, seed)
    bits = None if case["causal"] else _tree(N, seed)[2]
    return dict(q=_normal(g, (B, N, cfg.q_heads, cfg.head_dim), dt, 1.0), k=kv[0], v=kv[1], lens=lens, bits=bits,
                seq_len=torch.tensor(lens, dtype=torch.int32, device=DEV), anc=None if bits is None else _masks(bits),
                cfg=cfg, nodes=N)


def _verify_inputs(case, seed):
    cfg, dt, B, N, P = _cfg(case), _dtype(case), case["batch"], case["nodes"], case["prefix"]
    g = _gen(seed, 2)
    cache = KVCache(cfg, B, P + N + 80, dtype=dt, device=DEV)
    lens = _lengths(B, P, seed)
    cache.kv.normal_(0.0, 0.7, generator=g)
    cache.seq_len.copy_(torch.tensor(lens, dtype=torch.int32))
    _, dep, bits = _tree(N, seed)
    tokens = torch.randint(0, cfg.vocab, (B, N), dtype=torch.int32, device=DEV, generator=g)
    return dict(cfg=cfg, cache=cache, lens=lens, tokens=tokens, bits=bits, dep=dep, anc=_masks(bits),
                pos=torch.tensor(dep, dtype=torch.int32, device=DEV), err=torch.zeros(1, dtype=torch.int32, device=DEV))


def _prefill_inputs(case, seed):
    cfg, B, P = _cfg(case), case["batch"], case["prompt"]
    lens = _lengths(B, P, seed)
    lens[0] = P
    ids = torch.randint(0, cfg.vocab, (B, P), dtype=torch.int32, device=DEV, generator=_gen(seed, 2))
    return cfg, lens, ids


class _NoEos:
    pad_token_id, eos_token_id = 0, -1


def prepare(case, seed):
    kind, dt = case["kind"], _dtype(case)
    s = dict(case=case)
    if kind == "draw":
        s.update(logits=_logits(case["rows"], case["vocab"], dt, seed), seed=int(seed) + 17,
                 ids=torch.arange(case["rows"], dtype=torch.int32, device=DEV))
    elif kind == "attention":
        s.update(_attention_inputs(case, seed))
        s["out"] = torch.empty_like(s["q"])
    elif kind == "verify":
        s.update(_verify_inputs(case, seed))
        s["model"] = TargetModel(s["cfg"], _weights(s["cfg"], dt, seed), dtype=dt, device=DEV)
    elif kind == "prefill":
        cfg, lens, ids = _prefill_inputs(case, seed)
        s.update(ids=ids, lens=lens, model=TargetModel(cfg, _weights(cfg, dt, seed), dtype=dt, device=DEV),
                 cache=KVCache(cfg, case["batch"], case["prompt"] + 80, dtype=dt, device=DEV))
    elif kind in ("proposals", "chain"):
        cfg = _cfg(case)
        g = _gen(seed, 2)
        s["model"] = TargetModel(cfg, _weights(cfg, dt, seed), dtype=dt, device=DEV)
        s["heads"] = _heads(cfg, case.get("heads", 1), seed)
        if kind == "proposals":
            s["hidden"] = _normal(g, (case["batch"], cfg.hidden), dt, 1.0)
        else:
            R = case["batch"] * case["parents"]
            s["states"] = _normal(g, (R, cfg.hidden), torch.float32, 1.0)
            s["children"] = torch.randint(0, cfg.vocab, (R * case["kmax"],), dtype=torch.int32, device=DEV, generator=g)
            s["of"] = torch.arange(R * case["kmax"], device=DEV) // case["kmax"]
    elif kind == "walk":
        s.update(_walk_inputs(case, seed))
    else:
        cfg = MODELS[case["model"]]()
        g = _gen(seed, 2)
        P = case["prefix"]
        lens = _lengths(case["prompts"], P, seed)
        lens[0] = P
        ids = torch.randint(0, cfg.vocab, (case["prompts"], P), device=DEV, generator=g)
        mask = torch.arange(P, device=DEV)[None, :] >= P - torch.tensor(lens, device=DEV)[:, None]  # left padding
        model = TargetModel(cfg, _weights(cfg, dt, seed), dtype=dt, device=DEV)
        conf = FlashMedusaConfig(num_medusa_heads=3, tree_mode="fixed", max_tree_nodes_per_seq=16, max_tree_depth=4,
                                 fixed_tree_topk_by_depth=(4, 3, 2), temperature=1.0, top_p=0.95, noise_seed=int(seed) + 2)
        s.update(ids=ids, mask=mask, decoder=FlashMedusaDecoder(model, _heads(cfg, 3, seed), _NoEos(), conf))
    return s


def _walk_inputs(case, seed):
    """A verified tree whose hidden states point at known tokens: most steps at a child's token, some at
    another one, so that rows leave the walk at different depths, as in a rollout with trained heads."""
    cfg, dt, B, P = _cfg(case), _dtype(case), case["batch"], case["prefix"]
    ks = [int(k) for k in case["tree"].split(",")]
    par, dep, frontier = [-1], [0], [0]
    for k in ks:
        nxt = []
        for p in frontier:
            for _ in range(k):
                par.append(p)
                dep.append(dep[p] + 1)
                nxt.append(len(par) - 1)
        frontier = nxt
    N = len(par)
    g = _gen(seed, 2)
    w = {"embed": None, "layers": [], "final_norm": None, "lm_head": _normal(g, (cfg.vocab, cfg.hidden), dt, 0.02)}
    w["embed"] = w["lm_head"]
    model = TargetModel(dataclasses.replace(cfg, num_layers=0), w, dtype=dt, device=DEV)
    rnd = random.Random(int(seed) + 5)
    tok = np.array([rnd.sample(range(cfg.vocab), N) for _ in range(B)], dtype=np.int64)
    aim = np.zeros((B, N), dtype=np.int64)
    for b in range(B):
        for n in range(N):
            kids = [c for c in range(N) if par[c] == n]
            aim[b, n] = tok[b, rnd.choice(kids)] if kids and rnd.random() < 0.8 else rnd.randrange(cfg.vocab)
    tok_d = torch.from_numpy(tok.astype(np.int32)).to(DEV)
    noise = _normal(g, (B, N, cfg.hidden), torch.float32, 0.3)
    hidden = (w["lm_head"].index_select(0, torch.from_numpy(aim.reshape(-1)).to(DEV)).view(B, N, -1).float() * 40 + noise).to(dt)
    cache = KVCache(cfg, B, P + N + 80, dtype=dt, device=DEV)
    cache.kv.normal_(0.0, 0.7, generator=g)
    lens = _lengths(B, P, seed)
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    D = len(ks)
    return dict(cfg=cfg, model=model, hidden=hidden, tokens=tok_d, cache=cache, seq=seq, steps=D, nodes=N, seed=int(seed) + 9,
                parents=torch.tensor([par] * B, dtype=torch.int32, device=DEV),
                n_nodes=torch.full((B,), N, dtype=torch.int32, device=DEV), ids=torch.arange(B, dtype=torch.int32, device=DEV),
                err=torch.zeros(1, dtype=torch.int32, device=DEV),
                logits=torch.zeros(D, B, cfg.vocab, dtype=dt, device=DEV))


# ------------------------------------------------------------------ one pass
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "draw":
        return K.sample_tokens(s["logits"], seed=s["seed"], step=3, seq_ids=s["ids"], temperature=c["temperature"],
                               top_k=c["top_k"] or None, top_p=c["top_p"])
    if kind == "attention":
        cfg = s["cfg"]
        return K.tree_attention(s["q"], s["k"], s["v"], seq_len=s["seq_len"], anc=s["anc"], num_nodes=s["nodes"],
                                q_heads=cfg.q_heads, kv_heads=cfg.kv_heads, head_dim=cfg.head_dim, out=s["out"])
    if kind == "verify":
        h = s["model"].forward(s["tokens"], s["cache"], pos_offset=s["pos"], anc=s["anc"], err_flag=s["err"], graph=True)
        return dict(hidden=h, kv=s["cache"].kv, err=s["err"])
    if kind == "prefill":
        h = s["model"].prefill(s["ids"], s["cache"], lengths=s["lens"])
        return dict(last=h, kv=s["cache"].kv, seq_len=s["cache"].seq_len)
    if kind == "proposals":
        proj = s["heads"].project_all(s["hidden"], c["heads"])
        _, tok, score, stats = s["model"].logits_topk(proj, c["kmax"], stats=True)
        return dict(proj=proj, tokens=tok, scores=score, stats=stats)
    if kind == "chain":
        m = s["model"]
        _, tok, score, stats = m.logits_topk(s["states"].to(m.dtype), c["kmax"], stats=True, sanitize=True)
        nxt = s["heads"].chain_next_state(s["states"].index_select(0, s["of"]), s["children"], m.embed_weight)
        return dict(tokens=tok, scores=score, stats=stats, states=nxt)
    if kind == "walk":
        return _walk(s)
    dec = s["decoder"]
    r = dec.start(s["ids"], s["mask"], repeated_generate_nums=c["repeats"], max_length=c["prefix"] + 256)
    for _ in range(c["rounds"] - 1):
        dec.step(r)
    dec.flush(r)
    out = dict(logits=r.logits, hidden=r.hidden, seq_len=r.seq)
    dec.finish(r)
    width = max(len(t) for t in r.generated)
    out["tokens"] = np.array([t + [-1] * (width - len(t)) for t in r.generated], dtype=np.int64)
    return out


def _walk(s):
    m, B, N, D = s["model"], s["tokens"].shape[0], s["nodes"], s["steps"]
    walk = K.walk_begin(s["tokens"], s["parents"], s["n_nodes"], acc_stride=D + 1)
    parts = m.walk_parts(B, s["hidden"])
    K.walk_rows(walk, N)
    for t in range(D):
        m.logits(s["hidden"], row_index=walk["row_index"], row_active=walk["row_active"], out=s["logits"][t], parts=parts)
        K.walk_step(walk, s["logits"][t], s["tokens"], s["parents"], s["n_nodes"], walk_step=t, parts=parts, next_rows=True,
                    seed=s["seed"], step=3, seq_ids=s["ids"], err_flag=s["err"])
    fin = K.accept_finalize(walk, s["seq"], max_length=1 << 20, eos_token_id=None)
    s["cache"].gather_path(s["seq"], walk["acc_nodes"], walk["acc_len"], N, err_flag=s["err"])
    return dict(tokens=walk["acc_tokens"], nodes=walk["acc_nodes"], length=walk["acc_len"], last=walk["last_node"],
                finished=fin, logits=s["logits"], kv=s["cache"].kv, err=s["err"])


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    kind = case["kind"]
    fp32 = _dtype(case) == torch.float32
    if kind == "draw":
        return "exact"            # an integer rule: every implementation draws the same token
    if kind == "rollout":
        return {"rel": 2e-5, "max": 2e-3, "differ": 0.01}
    if kind == "walk":
        return {"rel": 1e-2, "max": 0.1}
    if kind in ("proposals", "chain"):
        # candidates whose bf16 logits lie a rounding apart may change places
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    if kind == "attention":
        # 2.3e-3 off 64 bits in bf16
        return {"rel": 1e-5, "max": 1e-3} if fp32 else {"rel": 1e-2, "max": 0.1}
    # against 64 bits the bf16 layers are 0.8e-2 to 1.4e-2 off, the fp32 ones below 1e-5
    return {"rel": 2e-5, "max": 2e-3} if fp32 else {"rel": 2.5e-2, "max": 0.3}


# ------------------------------------------------------------------ the same in 64 bits
def _attend64(q, k, v, lens, bits, scale):
    """q [B, N, Hq, d], k / v [B, Hkv, S, d]: softmax attention, one sequence at a time."""
    B, N, Hq, d = q.shape
    Hkv = k.shape[1]
    G = Hq // Hkv
    if bits is None:
        see = torch.tril(torch.ones(N, N, dtype=torch.bool, device=q.device))
    else:
        see = torch.tensor([[(int(w) >> m) & 1 for m in range(N)] for w in bits], dtype=torch.bool, device=q.device)
    out = torch.empty(B, N, Hq, d, dtype=torch.float64, device=q.device)
    for b in range(B):
        L = lens[b]
        kb, vb = k[b, :, :L + N].double(), v[b, :, :L + N].double()
        allow = torch.cat([torch.ones(N, L, dtype=torch.bool, device=q.device), see], 1)
        for h in range(Hkv):
            qb = q[b, :, h * G:(h + 1) * G].double().transpose(0, 1).reshape(G * N, d)
            sc = ((qb @ kb[h].t().contiguous()) * scale).view(G, N, L + N).masked_fill_(~allow, float("-inf"))
            o = torch.softmax(sc, -1).view(G * N, L + N) @ vb[h]
            out[b, :, h * G:(h + 1) * G] = o.view(G, N, d).transpose(0, 1)
    return out


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _forward64(cfg, w, tokens, kv, lens, dep, bits):
    """Decoder layers over tokens [B, N] after lens[b] committed tokens; writes kv [L, 2, B, Hkv, S, d] (float64)."""
    B, N = tokens.shape
    d, Hq, Hkv = cfg.head_dim, cfg.q_heads, cfg.kv_heads
    inv = (1.0 / (float(cfg.rope_theta) ** (torch.arange(0, d, 2, dtype=torch.int64).float() / d))).double().to(DEV)
    pos = torch.tensor(lens, device=DEV)[:, None] + torch.tensor(dep, device=DEV)[None, :]
    ang = pos.double()[:, :, None] * inv
    cos, sin = ang.cos()[:, :, None, :], ang.sin()[:, :, None, :]

    def rope(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = w["embed"].index_select(0, tokens.reshape(-1).long()).double()
    for l, lw in enumerate(w["layers"]):
        qkv = _norm64(x, lw["input_norm"], cfg.rms_eps) @ lw["qkv_w"].double().t().contiguous()
        if lw["qkv_b"] is not None:
            qkv = qkv + lw["qkv_b"].double()
        qkv = qkv.view(B, N, Hq + 2 * Hkv, d)
        q, k, v = rope(qkv[:, :, :Hq]), rope(qkv[:, :, Hq:Hq + Hkv]), qkv[:, :, Hq + Hkv:]
        for b in range(B):
            kv[l, 0, b, :, lens[b]:lens[b] + N] = k[b].transpose(0, 1)
            kv[l, 1, b, :, lens[b]:lens[b] + N] = v[b].transpose(0, 1)
        a = _attend64(q, kv[l, 0], kv[l, 1], lens, bits, 1 / math.sqrt(d))
        x = x + a.reshape(B * N, Hq * d) @ lw["o_w"].double().t().contiguous()
        gu = _norm64(x, lw["post_norm"], cfg.rms_eps) @ lw["gate_up_w"].double().t().contiguous()
        gate, up = gu.chunk(2, -1)
        x = x + (torch.nn.functional.silu(gate) * up) @ lw["down_w"].double().t().contiguous()
    return _norm64(x, w["final_norm"], cfg.rms_eps).view(B, N, cfg.hidden)


def _lm64(x, w):
    """x . w^T in 64 bits, the weight taken a slab at a time."""
    return torch.cat([x @ s.double().t().contiguous() for s in w.split(16384)], -1)


def _top64(lg, k):
    return lg.topk(k, -1)[0], torch.stack([lg.max(-1)[0], torch.logsumexp(lg, -1)], -1)


def exact(case, seed):
    kind, dt = case["kind"], _dtype(case)
    with torch.no_grad():
        if kind == "attention":
            s = _attention_inputs(case, seed)
            return _attend64(s["q"], s["k"], s["v"], s["lens"], s["bits"], 1 / math.sqrt(s["cfg"].head_dim))
        if kind == "verify":
            s = _verify_inputs(case, seed)
            kv = s["cache"].kv.double()
            h = _forward64(s["cfg"], _weights(s["cfg"], dt, seed), s["tokens"], kv, s["lens"], s["dep"], s["bits"])
            return dict(hidden=h, kv=kv, err=None)
        if kind == "prefill":
            cfg, lens, ids = _prefill_inputs(case, seed)
            B, P = ids.shape
            kv = torch.zeros(cfg.num_layers, 2, B, cfg.kv_heads, P + 80, cfg.head_dim, dtype=torch.float64, device=DEV)
            h = _forward64(cfg, _weights(cfg, dt, seed), ids, kv, [0] * B, list(range(P)), None)
            return dict(last=h[torch.arange(B, device=DEV), torch.tensor(lens, device=DEV) - 1], kv=kv, seq_len=None)
        if kind == "proposals":
            s = prepare(case, seed)
            x = s["hidden"].double()
            proj = []
            for hd in list(s["heads"].heads)[:case["heads"]]:
                n = torch.nn.functional.layer_norm(x, (x.shape[1],), hd.norm.weight.double(), hd.norm.bias.double(), hd.norm.eps)
                fc = n @ hd.fc.weight.to(dt).double().t().contiguous() + hd.fc.bias.to(dt).double()
                proj.append(x + torch.nn.functional.silu(fc))
            proj = torch.cat(proj)
            score, stats = _top64(_lm64(proj, s["model"].lm_head_weight), case["kmax"])
            return dict(proj=proj, tokens=None, scores=score, stats=stats)
        if kind == "chain":
            s = prepare(case, seed)
            m, cell = s["model"], s["heads"].chain_cell
            score, stats = _top64(_lm64(s["states"].to(dt).double(), m.lm_head_weight), case["kmax"])
            ln = lambda t, n: torch.nn.functional.layer_norm(t, (t.shape[1],), n.weight.double(), n.bias.double(), n.eps)  # noqa: E731
            st = s["states"].index_select(0, s["of"]).double()
            em = m.embed_weight.index_select(0, s["children"].long()).double()
            mix = (ln(st, cell.state_norm) @ cell.state_proj.weight.double().t().contiguous()
                   + ln(em, cell.token_norm) @ cell.token_proj.weight.double().t().contiguous())
            delta = torch.nn.functional.silu(mix) @ cell.out_proj.weight.double().t().contiguous() + cell.out_proj.bias.double()
            return dict(tokens=None, scores=score, stats=stats, states=st + torch.sigmoid(cell.gate.double()) * delta)
    return None  # whole numbers (draws), or values that hang on the tokens drawn (walk, rollout)
