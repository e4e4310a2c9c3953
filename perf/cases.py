"""The calls whose speed matters to a program built on specfit_amd.

Every case is one public entry point (or the one short sequence of them that
a decoder layer runs) at sizes a Qwen3-30B-A3B-shaped target meets: one-token
decoding, the verification of a draft tree, and the prefill of a prompt.

    kind      entry points
    router    Qwen3MoeTopKRouterHip.forward
    attn      ops.tree_attention (the attention implementation of a layer)
    experts   Qwen3OffloadedExperts.forward over a GpuExpertCache
    norms     ops.rms_norm and ops.qk_norm_rope (what a layer runs before attention)
    record    ops.expert_decode (the receiving end of a coded expert transfer)
    layer     Qwen3AttentionHip.forward (a decoder layer's whole attention module)
"""
import math
import random

import numpy as np
import torch

HIDDEN, INTER, EXPERTS, TOP_K = 2048, 768, 128, 8   # one MoE block of Qwen3-30B-A3B
BIG_HIDDEN, BIG_INTER = 4096, 1536                  # one expert of Qwen3-235B-A22B
Q_HEADS, KV_HEADS, HEAD_DIM = 32, 4, 128
EPS = 1e-6
DEV = "cuda:0"


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # Routing of one decoded token: the smallest call of the path, all
        # latency and launches.
        dict(name="router_decode", kind="router", tokens=1, hidden=HIDDEN, experts=EXPERTS, top_k=TOP_K),
        # Routing of a prompt.
        dict(name="router_prefill", kind="router", tokens=2048, hidden=HIDDEN, experts=EXPERTS, top_k=TOP_K),
        # Attention of one decoded token over a long context.
        dict(name="attn_decode", kind="attn", queries=1, context=4096, mask="none",
             q_heads=Q_HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM),
        # Attention of a 60-node draft tree and its seed over a 1024-token
        # context, with the tree's ancestor mask: the verification forward.
        dict(name="attn_verify", kind="attn", queries=61, context=1024, mask="tree",
             q_heads=Q_HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM),
        # Attention of a whole prompt: causal, no earlier context.
        dict(name="attn_prefill", kind="attn", queries=4096, context=0, mask="none",
             q_heads=Q_HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM),
        # The routed experts of one decoded token, every expert resident
        # (the whole model fits the card's memory).
        dict(name="experts_decode", kind="experts", tokens=1, slots=EXPERTS, zipf=False,
             hidden=HIDDEN, inter=INTER, experts=EXPERTS),
        # A 16-token tree with every expert resident and uniform routing: the
        # resident workload of bench.py.
        dict(name="experts_verify", kind="experts", tokens=16, slots=EXPERTS, zipf=False,
             hidden=HIDDEN, inter=INTER, experts=EXPERTS),
        # A prompt through one layer's resident experts.
        dict(name="experts_prefill", kind="experts", tokens=2048, slots=EXPERTS, zipf=False,
             hidden=HIDDEN, inter=INTER, experts=EXPERTS),
        # A 64-token tree through a 24-slot cache with Zipf routing, misses
        # arriving as coded records: the default workload of bench.py (bound
        # by the host link).
        dict(name="experts_offload", kind="experts", tokens=64, slots=24, zipf=True,
             hidden=HIDDEN, inter=INTER, experts=EXPERTS),
        # The norms and the rotary embedding of a layer for one tree.
        dict(name="norms_verify", kind="norms", tokens=61),
        # One expert's coded record into its slot: every miss pays this.
        dict(name="record_decode", kind="record", values=3 * HIDDEN * INTER, spread="normal"),
        # A decoder layer's whole attention module (projections, norms, rotary
        # embedding, cache update, attention) in the verification forward.
        dict(name="layer_verify", kind="layer", queries=61, context=1024, mask="tree",
             q_heads=Q_HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM),
    ]


def _log_uniform(rng: random.Random, low: int, high: int) -> int:
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng: random.Random):
    kind = rng.choice(["router", "attn", "attn", "attn", "experts", "experts", "experts", "norms",
                       "record"])
    if kind == "router":
        return dict(kind=kind, tokens=_log_uniform(rng, 2, 2000), experts=EXPERTS, top_k=TOP_K,
                    hidden=rng.choice([HIDDEN, HIDDEN, BIG_HIDDEN]))
    if kind == "attn":
        heads, kv, dim = rng.choice([(Q_HEADS, KV_HEADS, HEAD_DIM)] * 3 + [(64, 4, 128), (16, 4, 64)])
        phase = rng.choice(["decode", "tree", "prefill"])
        if phase == "decode":
            return dict(kind=kind, queries=1, context=_log_uniform(rng, 16, 16384), mask="none",
                        q_heads=heads, kv_heads=kv, head_dim=dim)
        if phase == "tree":
            return dict(kind=kind, queries=_log_uniform(rng, 4, 129), context=_log_uniform(rng, 16, 8192),
                        mask="tree", q_heads=heads, kv_heads=kv, head_dim=dim)
        # A prompt, or a later chunk of one: Q new tokens after the context.
        queries = _log_uniform(rng, 64, 2500)
        context = 0 if rng.random() < 0.6 else rng.randrange(1, 4097 - queries)
        return dict(kind=kind, queries=queries, context=context, mask="none", q_heads=heads,
                    kv_heads=kv, head_dim=dim)
    if kind == "experts":
        if rng.random() < 0.2:
            return dict(kind=kind, tokens=_log_uniform(rng, 1, 512), slots=32, zipf=False,
                        hidden=BIG_HIDDEN, inter=BIG_INTER, experts=32)
        return dict(kind=kind, tokens=_log_uniform(rng, 1, 2048), slots=EXPERTS,
                    zipf=rng.random() < 0.4, hidden=HIDDEN, inter=INTER, experts=EXPERTS)
    if kind == "norms":
        return dict(kind=kind, tokens=_log_uniform(rng, 1, 4096))
    return dict(kind=kind, values=_log_uniform(rng, 4096, 3 * BIG_HIDDEN * BIG_INTER),
                spread=rng.choice(["normal", "normal", "wide"]))


# ----------------------------------------------------------------- inputs --
def _gen(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + stream)


def _normal(shape, gen, std: float = 1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0.0, std, generator=gen)


def _zipf_bias(experts: int, rng: np.random.Generator) -> np.ndarray:
    p = np.arange(1, experts + 1, dtype=np.float64) ** -1.1
    return rng.permutation(np.log(p / p.sum()))


def _routes(tokens: int, experts: int, zipf: bool, seed: int):
    """(index int64 [T, 8], weight fp32 [T, 8]) of a top-8 softmax router whose
    logits are N(0, 0.9) (N(0, 1) states through N(0, 0.02) rows of 2048),
    plus a Zipf(1.1) popularity bias when asked, renormalised."""
    rng = np.random.default_rng(seed + 17)
    logits = rng.normal(0.0, 0.9, (tokens, experts))
    if zipf:
        logits = logits + _zipf_bias(experts, rng)
    idx = np.argsort(-logits, axis=1, kind="stable")[:, :TOP_K]
    top = np.exp(np.take_along_axis(logits, idx, axis=1))
    return idx.astype(np.int64), (top / top.sum(axis=1, keepdims=True)).astype(np.float32)


def _expert_weights(case, seed: int) -> torch.Tensor:
    return _normal((case["experts"], 3 * case["inter"] * case["hidden"]), _gen(seed, 1), 0.02)


def _expert_inputs(case, seed: int):
    idx, weight = _routes(case["tokens"], case["experts"], case["zipf"], seed)
    hidden = _normal((case["tokens"], case["hidden"]), _gen(seed, 2))
    return (hidden, torch.from_numpy(idx).to(DEV),
            torch.from_numpy(weight).to(DEV).to(torch.bfloat16))


def _tree_parents(queries: int, depth: int, rng: np.random.Generator) -> np.ndarray:
    """parent[i] < i of node i (0 is the seed), about queries/depth nodes a level."""
    parents = np.zeros(queries, dtype=np.int64)
    per = max(1, math.ceil((queries - 1) / depth))
    for i in range(1, queries):
        level = (i - 1) // per
        parents[i] = 0 if level == 0 else 1 + (level - 1) * per + rng.integers(per)
    return parents


def _attn_mask(case, seed: int):
    if case["mask"] == "none":
        return None
    q, ctx = case["queries"], case["context"]
    parents = _tree_parents(q, 6, np.random.default_rng(seed + 29))
    mask = np.zeros((q, ctx + q), dtype=bool)
    mask[:, :ctx] = True
    for i in range(q):
        mask[i, ctx + i] = True
        if i:
            mask[i, ctx:] |= mask[parents[i], ctx:]
    return torch.from_numpy(mask).to(DEV)[None, None]


def _attn_inputs(case, seed: int):
    q, s, d = case["queries"], case["context"] + case["queries"], case["head_dim"]
    gen = _gen(seed, 3)
    return (_normal((1, case["q_heads"], q, d), gen), _normal((1, case["kv_heads"], s, d), gen),
            _normal((1, case["kv_heads"], s, d), gen), _attn_mask(case, seed))


def _norm_inputs(case, seed: int):
    t, gen = case["tokens"], _gen(seed, 4)
    x = _normal((1, t, HIDDEN), gen, 2.0)
    weight = _normal((HIDDEN,), gen, 0.1) + 1.0
    qkv = _normal((1, t, (Q_HEADS + 2 * KV_HEADS) * HEAD_DIM), gen, 1.5)
    wq, wk = _normal((HEAD_DIM,), gen, 0.1) + 1.0, _normal((HEAD_DIM,), gen, 0.1) + 1.0
    inv = 1e6 ** (-torch.arange(0, HEAD_DIM, 2, device=DEV, dtype=torch.float64) / HEAD_DIM)
    angle = (1024 + torch.arange(t, device=DEV, dtype=torch.float64))[:, None] * inv
    angle = torch.cat([angle, angle], dim=-1)[None]
    return x, weight, qkv, wq, wk, angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)


def _record_values(case, seed: int) -> torch.Tensor:
    gen = _gen(seed, 5)
    v = torch.empty(case["values"], dtype=torch.float32, device=DEV).normal_(0.0, 0.02, generator=gen)
    if case["spread"] == "wide":  # a few large and many tiny weights: more codes of the later levels
        v *= torch.empty_like(v).normal_(0.0, 1.0, generator=gen).exp_()
    return v.to(torch.bfloat16)


class _State(dict):
    """What the program holds; a cache gives its slots back with it."""

    def __del__(self):
        for cache in self.get("caches", ()):
            cache.close()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "router":
        from specfit_amd.runtime import Qwen3MoeTopKRouterHip

        gen = _gen(seed, 0)
        router = Qwen3MoeTopKRouterHip(num_experts=case["experts"], hidden_size=case["hidden"],
                                       top_k=case["top_k"], norm_topk_prob=True, device=DEV)
        router.weight.copy_(_normal((case["experts"], case["hidden"]), gen, 0.02))
        return _State(kind=kind, router=router, hidden=_normal((case["tokens"], case["hidden"]), gen))
    if kind == "attn":
        q, k, v, mask = _attn_inputs(case, seed)
        return _State(kind=kind, q=q, k=k, v=v, mask=mask, scale=case["head_dim"] ** -0.5)
    if kind == "experts":
        return _prepare_experts(case, seed)
    if kind == "norms":
        x, weight, qkv, wq, wk, cos, sin = _norm_inputs(case, seed)
        nq, nk = Q_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
        t = case["tokens"]
        return _State(kind=kind, x=x, weight=weight, wq=wq, wk=wk, cos=cos, sin=sin,
                      q=qkv[..., :nq].view(1, t, Q_HEADS, HEAD_DIM),
                      k=qkv[..., nq:nq + nk].view(1, t, KV_HEADS, HEAD_DIM))
    if kind == "record":
        from specfit_amd.codec import encode_record

        values = _record_values(case, seed)
        record, counts, table = encode_record(values, force=True)
        return _State(kind=kind, record=record, counts=counts, table=table, out=torch.empty_like(values))
    return _prepare_layer(case, seed)


def _prepare_experts(case, seed):
    from specfit_amd.codec import CompressedExperts
    from specfit_amd.runtime import ExpertKey, GpuExpertCache, Qwen3OffloadedExperts

    n = case["experts"]
    device_weights = _expert_weights(case, seed)
    host = torch.empty(device_weights.shape, dtype=torch.bfloat16, pin_memory=True)
    host.copy_(device_weights)
    sources = {ExpertKey(0, e): host[e] for e in range(n)}
    image = None
    if case["slots"] < n:
        image = CompressedExperts.encode({ExpertKey(0, e): device_weights[e] for e in range(n)}, device=DEV)
    del device_weights
    cache = GpuExpertCache(sources, slot_count=case["slots"], device=DEV, adopt_pinned_sources=True,
                           compressed_sources=image)
    module = Qwen3OffloadedExperts(layer_id=0, cache=cache, hidden_size=case["hidden"],
                                   intermediate_size=case["inter"], execution_policy="resident_first",
                                   h2d_prefetch=True)
    hidden, idx, weight = _expert_inputs(case, seed)
    if case["slots"] == n:
        for e in range(n):
            with cache.acquire(ExpertKey(0, e)) as lease:
                lease.wait()
    else:  # the cache as earlier trees of the same distribution leave it
        for cycle in range(1, 4):
            module(*_expert_inputs(case, seed + 100 * cycle))
    torch.cuda.synchronize()
    return _State(kind="experts", module=module, hidden=hidden, idx=idx, weight=weight, caches=(cache,))


def _layer_inputs(case, seed: int):
    """Weights, hidden states, rotary tables, cached keys and values, mask."""
    gen, d = _gen(seed, 6), HEAD_DIM
    w = {"q_proj": _normal((Q_HEADS * d, HIDDEN), gen, 0.02), "k_proj": _normal((KV_HEADS * d, HIDDEN), gen, 0.02),
         "v_proj": _normal((KV_HEADS * d, HIDDEN), gen, 0.02), "o_proj": _normal((HIDDEN, Q_HEADS * d), gen, 0.02),
         "q_norm": _normal((d,), gen, 0.1) + 1.0, "k_norm": _normal((d,), gen, 0.1) + 1.0}
    hidden = _normal((1, case["queries"], HIDDEN), gen)
    position = case["context"] + torch.arange(case["queries"], device=DEV, dtype=torch.float64) // 10
    inv = 1e6 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    angle = torch.cat([position[:, None] * inv] * 2, dim=-1)[None]
    kv = [_normal((1, KV_HEADS, case["context"], d), gen) for _ in range(2)]
    return w, hidden, angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16), kv, _attn_mask(case, seed)


def _prepare_layer(case, seed):
    from transformers import DynamicCache, Qwen3MoeConfig
    from transformers.models.qwen3_moe.modeling_qwen3_moe import Qwen3MoeAttention

    from specfit_amd.runtime import register_tree_attention
    from specfit_amd.runtime.qwen3_attention import Qwen3AttentionHip
    from specfit_amd.runtime.qwen3_norm import Qwen3RMSNormHip
    from specfit_amd.workloads import QWEN3_30B_A3B_MODEL

    config = Qwen3MoeConfig(**dict(QWEN3_30B_A3B_MODEL, num_hidden_layers=1))
    config._attn_implementation = register_tree_attention()
    weights, hidden, cos, sin, (k, v), mask = _layer_inputs(case, seed)
    with torch.device("meta"):
        module = Qwen3MoeAttention(config, layer_idx=0)
    for name, value in weights.items():
        getattr(module, name).weight = torch.nn.Parameter(value, requires_grad=False)
    for name in ("q_norm", "k_norm"):
        setattr(module, name, Qwen3RMSNormHip.from_module(getattr(module, name)))
    cache = DynamicCache()
    cache.update(k, v, 0)
    return _State(kind="layer", module=Qwen3AttentionHip.from_module(module).eval(), hidden=hidden,
                  rotary=(cos, sin), mask=mask, cache=cache)


# -------------------------------------------------------------------- run --
@torch.inference_mode()
def run(state):
    from specfit_amd import ops

    kind = state["kind"]
    if kind == "router":
        logits, weight, idx = state["router"](state["hidden"])
        return {"logits": logits, "weight": weight, "index": idx}
    if kind == "attn":
        return ops.tree_attention(state["q"], state["k"], state["v"], state["mask"], state["scale"])
    if kind == "experts":
        return state["module"](state["hidden"], state["idx"], state["weight"])
    if kind == "norms":
        normed = ops.rms_norm(state["x"], state["weight"], EPS)
        q, k = ops.qk_norm_rope(state["q"], state["k"], state["wq"], state["wk"], EPS, state["cos"],
                                state["sin"])
        return {"normed": normed, "q": q, "k": k}
    if kind == "record":
        ops.expert_decode(state["record"], state["counts"], state["table"], state["out"])
        return state["out"]
    out, _ = state["module"](state["hidden"], state["rotary"], state["mask"], past_key_values=state["cache"])
    state["cache"].crop(-state["hidden"].shape[1])
    return out


# ------------------------------------------------------------------- work --
def _distinct(case) -> int:
    """Distinct experts of one pass (routes of one seed stand for all)."""
    return len(np.unique(_routes(case["tokens"], case["experts"], case["zipf"], 0)[0]))


def _attn_pairs(queries: int, context: int, mask: str) -> int:
    if mask == "tree":  # the context and a node's few ancestors
        return queries * (context + min(queries, 4))
    return queries * context + queries * (queries + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "router":
        t, h, e, k = case["tokens"], case["hidden"], case["experts"], case["top_k"]
        return {"bytes": 2 * h * (e + t) + t * (2 * e + 10 * k), "flops": 2 * t * h * e}
    if kind == "attn":
        q, ctx, d = case["queries"], case["context"], case["head_dim"]
        mask = q * (q + ctx) if case["mask"] == "tree" else 0
        return {"bytes": 4 * q * case["q_heads"] * d + 4 * (q + ctx) * case["kv_heads"] * d + mask,
                "flops": 4 * case["q_heads"] * d * _attn_pairs(q, ctx, case["mask"])}
    if kind == "experts":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        return {"bytes": _distinct(case) * 6 * h * i + 4 * t * h + 10 * t * TOP_K,
                "flops": 6 * h * i * t * TOP_K}
    if kind == "norms":
        t = case["tokens"]
        heads = (Q_HEADS + KV_HEADS) * HEAD_DIM
        return {"bytes": 4 * t * (HIDDEN + heads + HEAD_DIM), "flops": 8 * t * (HIDDEN + 2 * heads)}
    if kind == "record":  # about 10.74 bits a value in, 16 out
        return {"bytes": case["values"] * 27 // 8, "flops": 0}
    q, ctx = case["queries"], case["context"]
    weights = HIDDEN * (2 * Q_HEADS + 2 * KV_HEADS) * HEAD_DIM
    return {"bytes": 2 * weights + 4 * q * HIDDEN + 4 * (q + ctx) * KV_HEADS * HEAD_DIM + q * (q + ctx),
            "flops": 2 * q * weights + 4 * Q_HEADS * HEAD_DIM * _attn_pairs(q, ctx, case["mask"])}


# -------------------------------------------------------------- tolerance --
def tolerance(case):
    kind = case["kind"]
    if kind in ("router", "record"):
        # Routing (logits, weights, indices) has a fixed summation order that
        # the CPU oracle shares, and the coding is lossless.
        return "exact"
    # The others: about four times what plain torch implementations with the
    # same roundings and other summation orders differ by.
    if kind == "attn":
        # 3.0e-3 and 6.1e-2 (bf16 probabilities of an unshifted softmax).
        return {"rel": 1.2e-2, "max": 0.25}
    if kind == "experts":
        # 3.6e-4 and 1.3e-2 (torch matmuls; equal bits at some sizes).
        return {"rel": 1.5e-3, "max": 0.05}
    if kind == "norms":
        # Equal bits; another order of the sum of squares moves single values
        # by one bf16 step (7.8e-3), through two roundings by two.
        return {"rel": 1e-3, "max": 2e-2}
    # 3.4e-3 and 1.5e-2 (torch's scaled dot product attention in the same module).
    return {"rel": 1.4e-2, "max": 6e-2}


# ------------------------------------------------------------------ exact --
def _exact_norm(t, w):
    t = t.double()
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_head(t, heads, w, cos, sin):
    """Normed and rotated heads [1, heads, T, 128] of a projection [1, T, heads * 128]."""
    t = _exact_norm(t.reshape(1, t.shape[1], heads, HEAD_DIM), w).transpose(1, 2)
    half = HEAD_DIM // 2
    turned = torch.cat([-t[..., half:], t[..., :half]], dim=-1)
    return t * cos.double()[:, None] + turned * sin.double()[:, None]


def _exact_attention(q, k, v, mask):
    queries, keys, heads, dim = q.shape[2], k.shape[2], q.shape[1], q.shape[3]
    if mask is None:
        last = torch.arange(keys - queries, keys, device=DEV)[:, None]
        allowed = torch.arange(keys, device=DEV)[None] <= last
    else:
        allowed = mask[0, 0]
    out = torch.empty((1, queries, heads, dim), dtype=torch.float64, device=DEV)
    for head in range(heads):
        kv = head // (heads // k.shape[1])
        scores = (q[0, head].double() @ k[0, kv].double().T) * dim ** -0.5
        probs = torch.softmax(scores.masked_fill(~allowed, -math.inf), dim=-1)
        out[0, :, head] = probs @ v[0, kv].double()
    return out


def _exact_layer(case, seed):
    w, hidden, cos, sin, (k_old, v_old), mask = _layer_inputs(case, seed)
    h = hidden.double()
    q, k, v = (h @ w[name].double().T for name in ("q_proj", "k_proj", "v_proj"))
    q = _exact_head(q, Q_HEADS, w["q_norm"], cos, sin)
    k = torch.cat([k_old.double(), _exact_head(k, KV_HEADS, w["k_norm"], cos, sin)], dim=2)
    v = torch.cat([v_old.double(), v.view(1, -1, KV_HEADS, HEAD_DIM).transpose(1, 2)], dim=2)
    out = _exact_attention(q, k, v, mask)
    return out.reshape(1, case["queries"], -1) @ w["o_proj"].double().T


def exact(case, seed):
    kind = case["kind"]
    if kind == "router":
        gen = _gen(seed, 0)
        weight = _normal((case["experts"], case["hidden"]), gen, 0.02).double()
        logits = _normal((case["tokens"], case["hidden"]), gen).double() @ weight.T
        top = torch.softmax(logits, dim=-1).topk(case["top_k"], dim=-1).values
        # Indices of equal bf16 logits go to the lower id, which 64 bits do not see.
        return {"logits": logits, "weight": top / top.sum(-1, keepdim=True), "index": None}
    if kind == "attn":
        return _exact_attention(*_attn_inputs(case, seed))
    if kind == "experts":
        packed = _expert_weights(case, seed)
        hidden, idx, weight = _expert_inputs(case, seed)
        h, i = case["hidden"], case["inter"]
        out = torch.zeros(hidden.shape, dtype=torch.float64, device=DEV)
        for e in range(case["experts"]):
            token, place = torch.nonzero(idx == e, as_tuple=True)
            if token.numel():
                w = packed[e].double()
                gate_up = hidden[token].double() @ w[:2 * i * h].view(2 * i, h).T
                act = torch.nn.functional.silu(gate_up[:, :i]) * gate_up[:, i:]
                rows = act @ w[2 * i * h:].view(h, i).T
                out.index_add_(0, token, rows * weight[token, place].double()[:, None])
        return out
    if kind == "norms":
        x, weight, qkv, wq, wk, cos, sin = _norm_inputs(case, seed)
        nq, nk = Q_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
        return {"normed": _exact_norm(x, weight), "q": _exact_head(qkv[..., :nq], Q_HEADS, wq, cos, sin),
                "k": _exact_head(qkv[..., nq:nq + nk], KV_HEADS, wk, cos, sin)}
    if kind == "record":
        return _record_values(case, seed).double()
    return _exact_layer(case, seed)
