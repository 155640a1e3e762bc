"""Performance cases: the work a decoding engine has this package do.

One case is one call (or one forward's worth of calls) through the public entry
points, with inputs made on the GPU from a seed.  Three kinds:

  op1   one MoE layer: ``tree_moe_forward``, or the engine's MoE hook
        (``make_moe_fn``: phase-1 routing, the demand observer, the GEMMs)
  attn  the tree attention of ``layers`` consecutive layers over one paged
        cache, as one forward calls it
  op4   ``fused_verify_commit``: verification of one draft tree and the commit
        of the accepted path into the paged cache

The listed cases cover a request from its prefill to its last verification
step; ``draw`` gives further cases of the same ranges.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from treemoe_spec_amd.kernels.op1_tree_moe import tree_moe_forward
from treemoe_spec_amd.kernels.op4_commit import fused_verify_commit
from treemoe_spec_amd.kernels.tree_attention import tree_attention
from treemoe_spec_amd.kv_cache import MixtralConfig, PagedKVCache
from treemoe_spec_amd.moe_adapter import make_moe_fn
from treemoe_spec_amd.workloads import op4_workload, random_tree

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
TAU = 0.05            # top1_threshold of the routing entry points
HEAD_DIM = 128
LARGEST_TOKENS = 6011


def _op1(name, tokens, hidden=4096, inter=14336, experts=8, budget=8, objective="mass",
         dtype="bf16", entry="forward", bias="none", accept="ones"):
    c = {"kind": "op1", "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts,
         "budget": budget, "objective": objective, "dtype": dtype, "entry": entry, "bias": bias,
         "accept": accept}
    return {"name": name, **c} if name else c


def _attn(name, nodes, seq, page=16, heads=32, kv_heads=8, layers=8):
    c = {"kind": "attn", "nodes": nodes, "seq": seq, "page": page, "heads": heads,
         "kv_heads": kv_heads, "layers": layers}
    return {"name": name, **c} if name else c


def _op4(name, nodes, vocab=32000, mode="greedy", dtype="bf16", seq=4096, page=16, depth=8,
         layers=32):
    c = {"kind": "op4", "nodes": nodes, "vocab": vocab, "mode": mode, "dtype": dtype, "seq": seq,
         "page": page, "depth": depth, "layers": layers}
    return {"name": name, **c} if name else c


def listed():
    return [
        # an autoregressive step: one token, two of the eight experts
        _op1("layer_1_token", 1),
        # the verification forward of a 64-node tree with every expert allowed
        _op1("layer_64_tree", 64),
        # the same tree through the engine's hook with a budget of 4 experts, skewed demand
        # and acceptance probabilities, and the objective that protects likely nodes
        _op1("layer_64_tree_hook_budget4", 64, budget=4, objective="critical_path", entry="hook",
             bias="normal", accept="uniform"),
        # a 64-node tree of the small layer that the tests and the CPU baseline use
        _op1("layer_64_tree_small", 64, hidden=1024, inter=3584),
        # prefill of a short prompt, odd length, in half precision
        _op1("layer_517_prefill_fp16", 517, dtype="fp16"),
        # prefill of 2048 tokens with Zipf-skewed experts
        _op1("layer_2048_prefill_skew", 2048, bias="zipf"),
        # prefill of a long prompt, odd length: the largest call
        _op1("layer_6011_prefill", LARGEST_TOKENS),
        # attention of a 64-node tree over 4096 cached positions
        _attn("attention_64_tree", 64, 4096),
        # attention of an autoregressive step over a long, odd-length cache
        _attn("attention_1_token", 1, 7777, page=64),
        # attention of a small odd tree soon after a short prompt
        _attn("attention_27_tree_short", 27, 333),
        # greedy verification of a 64-node tree and its commit
        _op4("verify_64_greedy", 64),
        # the same step in sampling mode (temperature 1, float32 logits)
        _op4("verify_64_sampling", 64, mode="sample", dtype="fp32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["op1", "op1", "op1", "op1", "attn", "attn", "op4"])
    if kind == "op1":
        # the Mixtral layer, one GPU's tensor-parallel share of it, or the small layer
        hidden, inter = rng.choice([(4096, 14336), (4096, 14336), (4096, 14336), (4096, 7168),
                                    (4096, 3584), (4096, 1792), (1024, 3584)])
        experts = rng.choice([8, 8, 8, 16]) if hidden == 1024 else 8
        return _op1(None, _log_int(rng, 1, LARGEST_TOKENS), hidden, inter, experts,
                    budget=rng.choice([2, 4, 6, 8, 8, 8]),
                    objective=rng.choice(["mass", "mass", "critical_path"]),
                    dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]),
                    entry=rng.choice(["forward", "hook"]),
                    bias=rng.choice(["none", "none", "normal", "zipf"]),
                    accept=rng.choice(["ones", "uniform"]))
    if kind == "attn":
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (8, 2)])
        return _attn(None, _log_int(rng, 1, 64), _log_int(rng, 16, 8000),
                     page=rng.choice([16, 64]), heads=heads, kv_heads=kv_heads,
                     layers=rng.choice([2, 8]))
    return _op4(None, _log_int(rng, 1, 64), rng.choice([32000, _log_int(rng, 1000, 131072)]),
                mode=rng.choice(["greedy", "greedy", "penalty", "sample"]),
                dtype=rng.choice(["bf16", "fp32"]), seq=_log_int(rng, 16, 4096),
                page=rng.choice([16, 64]), depth=rng.randint(2, 8))


# ------------------------------------------------------------------ inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _prepare_op1(case, seed):
    t, h, i, e = case["tokens"], case["hidden"], case["inter"], case["experts"]
    dt = DTYPES[case["dtype"]]
    g = _gen(seed)
    x = _normal(g, t, h, dtype=torch.float32)
    router = _normal(g, e, h, std=0.02, dtype=torch.float32)
    if case["bias"] == "normal":      # a per-expert bias, as a constant feature
        bias = torch.randn(e, generator=g, device=DEV) * 1.5
    elif case["bias"] == "zipf":
        bias = -1.2 * torch.log((torch.randperm(e, generator=g, device=DEV) + 1).float())
    else:
        bias = None
    if bias is not None:
        x[:, 0] = 1.0
        router[:, 0] = bias
    s = SimpleNamespace(x=x.to(dt), router=router.to(dt))
    s.w1 = _normal(g, e, i, h, std=0.02, dtype=dt)
    s.w3 = _normal(g, e, i, h, std=0.02, dtype=dt)
    s.w2 = _normal(g, e, h, i, std=0.02, dtype=dt)
    s.accept = torch.ones(t, device=DEV)
    if case["accept"] == "uniform":
        s.accept = torch.rand(t, generator=g, device=DEV)
    s.budget, s.objective = case["budget"], case["objective"]
    if case["entry"] == "hook":
        s.layer = SimpleNamespace(router=s.router, w1=s.w1, w2=s.w2, w3=s.w3)
        s.moe_fn = make_moe_fn(expert_budget=s.budget, routing_objective=s.objective,
                               tree_size=t, device=DEV)
        s.moe_fn.current_accept_prob = s.accept
        s.seen = {}
        s.moe_fn.demand_observer = lambda layer, demand: s.seen.update({layer: demand})
    return s


def _run_op1(s):
    if hasattr(s, "moe_fn"):
        out = s.moe_fn(s.x, s.layer, 0)
        return {"out": out, "demand": s.seen[0]}
    return {"out": tree_moe_forward(s.x, s.w1, s.w2, s.w3, s.router, s.accept, s.budget,
                                    routing_objective=s.objective)}


def _cache(g, case, nodes, extra):
    cfg = MixtralConfig(num_layers=case["layers"], num_kv_heads=case.get("kv_heads", 8),
                        num_heads=case.get("heads", 32), head_dim=HEAD_DIM)
    page, seq = case["page"], case["seq"]
    pages = -(-nodes // page) + -(-(seq + extra) // page) + 2
    kv = PagedKVCache(cfg, pages, device=DEV, page_size=page, tree_size=nodes)
    kv._ensure_capacity(seq)
    kv.seq_len = seq
    kv.k.normal_(0.0, 1.0, generator=g)
    kv.v.normal_(0.0, 1.0, generator=g)
    return kv


def _tree(seed, nodes, depth):
    return random_tree(torch.Generator().manual_seed(seed), nodes, depth)


def _prepare_attn(case, seed):
    g = _gen(seed)
    n = case["nodes"]
    parent = _tree(seed, n, 8)[0]
    mask = torch.eye(n, dtype=torch.bool)
    for j in range(1, n):           # a node sees itself and its ancestors
        mask[j] |= mask[parent[j]]
    s = SimpleNamespace(kv=_cache(g, case, n, 0), mask=mask.to(DEV))
    s.qkv = [(_normal(g, n, case["heads"], HEAD_DIM), _normal(g, n, case["kv_heads"], HEAD_DIM),
              _normal(g, n, case["kv_heads"], HEAD_DIM)) for _ in range(case["layers"])]
    return s


def _run_attn(s):
    outs = [tree_attention(q, k, v, s.kv, layer, s.mask) for layer, (q, k, v) in enumerate(s.qkv)]
    return {"out": outs, "k": s.kv.k, "v": s.kv.v}


def _prepare_op4(case, seed):
    g = _gen(seed)
    n, v, dt = case["nodes"], case["vocab"], DTYPES[case["dtype"]]
    s = SimpleNamespace(mode=case["mode"], depth=case["depth"], seq=case["seq"], seed=seed)
    s.kv = _cache(g, case, n, case["depth"] + 1)
    if case["mode"] == "sample":
        # the draft of a node is near the target's distribution at its parent, and its token
        # is drawn from that draft
        parent, s.children, _, _ = _tree(seed, n, case["depth"])
        logits = _normal(g, n, v, std=3.0, dtype=torch.float32).to(dt)
        at = torch.tensor([max(p, 0) for p in parent], device=DEV)
        s.draft = torch.softmax(logits.float()[at] + _normal(g, n, v, dtype=torch.float32), -1)
        s.tokens = torch.multinomial(s.draft, 1, generator=g).reshape(-1)
        s.parent = torch.tensor(parent, device=DEV)
        s.logits = logits
        s.generator = _gen(seed)
    else:
        w = op4_workload(n=n, vocab=v, max_depth=case["depth"], seed=seed, dtype=dt)
        s.logits, s.tokens, s.parent = w.logits.to(DEV), w.tokens.to(DEV), w.parent.to(DEV)
        s.children, s.draft, s.generator = w.children, None, None
        s.prev = torch.randint(0, v, (512,), generator=g, device=DEV)
    return s


def _run_op4(s):
    s.kv.seq_len = s.seq
    if s.mode == "sample":
        s.generator.manual_seed(s.seed)
        r = fused_verify_commit(s.logits, s.draft, s.tokens, s.parent, s.children, kv=s.kv,
                                temperature=1.0, generator=s.generator)
    elif s.mode == "penalty":
        # the penalty is applied in place to the step's fresh logits
        logits = s.logits.clone()
        r = fused_verify_commit(logits, None, s.tokens, s.parent, s.children, kv=s.kv,
                                rep_penalty=1.1, prev_tokens=s.prev, max_depth=s.depth)
        return {"slots": r.accepted_slots, "tokens": r.accepted_tokens, "bonus": r.bonus_token,
                "accepted": r.num_accepted, "seq_len": s.kv.seq_len, "k": s.kv.k, "v": s.kv.v,
                "logits": logits}
    else:
        r = fused_verify_commit(s.logits, None, s.tokens, s.parent, s.children, kv=s.kv,
                                max_depth=s.depth)
    return {"slots": r.accepted_slots, "tokens": r.accepted_tokens, "bonus": r.bonus_token,
            "accepted": r.num_accepted, "seq_len": s.kv.seq_len, "k": s.kv.k, "v": s.kv.v}


_PREPARE = {"op1": _prepare_op1, "attn": _prepare_attn, "op4": _prepare_op4}
_RUN = {"op1": _run_op1, "attn": _run_attn, "op4": _run_op4}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed), case["kind"]


def run(state):
    s, kind = state
    return _RUN[kind](s)


# -------------------------------------------------------------------- work --

def _active_experts(case):
    """Experts that `tokens` tokens reach: the expected number of distinct experts of two picks
    each, at most the budget (the skewed cases reach fewer, so this does not overstate the rate
    of the small ones by much)."""
    e, b = case["experts"], case["budget"]
    return min(b, e * (1.0 - (1.0 - 2.0 / e) ** case["tokens"]))


def work(case):
    if case["kind"] == "op1":
        t, h, i, e = case["tokens"], case["hidden"], case["inter"], case["experts"]
        return {"bytes": _active_experts(case) * 3 * h * i * 2 + 2 * t * h * 2 + e * h * 2 + 4 * t,
                "flops": 2 * t * h * e + 2 * t * 3 * 2 * h * i}
    if case["kind"] == "attn":
        n, s = case["nodes"], case["seq"]
        q, kv = case["heads"] * HEAD_DIM * 2, case["kv_heads"] * HEAD_DIM * 2
        # cached K and V, the tree's K and V in and out, q in, the context out
        return {"bytes": case["layers"] * (2 * s * kv + 4 * n * kv + 2 * n * q),
                "flops": case["layers"] * 4 * n * (s + n) * case["heads"] * HEAD_DIM}
    n, v = case["nodes"], case["vocab"]
    eb = 4 if case["dtype"] == "fp32" else 2
    row = case["layers"] * 8 * HEAD_DIM * 2
    depth = case["depth"] / 2
    if case["mode"] == "sample":   # the visited nodes' logits and draft rows
        data = depth * v * (eb + 4)
    else:
        data = n * v * eb
    return {"bytes": data + 4 * (depth + 1) * row, "flops": 0}


# ----------------------------------------------------------------- results --

def tolerance(case):
    if case["kind"] == "op1":
        # h and the output are rounded to 16 bits; another order of the fp32 sums moves some of
        # them by one unit (two GEMM kernels with different orders: 2e-4 to 4e-4 apart in bf16,
        # 9e-5 in fp16)
        return {"rel": 1.6e-3 if case["dtype"] == "bf16" else 4e-4}
    if case["kind"] == "attn":
        # the probabilities and the output are rounded to bf16 (other chunks of the keys:
        # 2.3e-3 to 3.2e-3 apart)
        return {"rel": 1.2e-2}
    return "exact"


def _exact_routing(s):
    """topk ids [T, 2] and gates [T, 2] (float64), demand [E]: the router's logits rounded to the
    activations' type as a linear layer returns them, everything after in 64 bits."""
    logits = (s.x.double() @ s.router.double().T).to(s.x.dtype)
    gates = torch.softmax(logits.double(), -1)
    e = gates.shape[1]
    accept = s.accept.double()
    demand = (accept[:, None] * gates).sum(0)

    def top2(g):
        first = g.argmax(-1)
        rest = g.scatter(1, first[:, None], -1.0)
        return first, rest.argmax(-1)

    crit = torch.zeros(e, dtype=torch.float64, device=gates.device)
    if s.objective == "critical_path":
        a, b = top2(gates)
        need = torch.full_like(gates, -math.inf)
        need.scatter_(1, a[:, None], accept[:, None])
        second = torch.where(accept >= TAU, accept, torch.full_like(accept, -math.inf))
        need.scatter_(1, b[:, None], second[:, None])
        crit = need.max(0).values
    order = sorted(range(e), key=lambda j: (-float(crit[j]), -float(demand[j]), j))
    keep = torch.zeros(e, dtype=torch.bool, device=gates.device)
    keep[torch.tensor(order[:s.budget], device=gates.device)] = True
    kept = torch.where(keep[None, :], gates, torch.zeros_like(gates))
    a, b = top2(kept)
    ids = torch.stack([a, b], 1)
    g = kept.gather(1, ids)
    g = g / g.sum(1, keepdim=True)
    low = s.accept < TAU
    g[low] = torch.tensor([1.0, 0.0], dtype=torch.float64, device=g.device)
    return ids, g, demand


def _exact_op1(s):
    ids, gates, demand = _exact_routing(s)
    out = torch.zeros(s.x.shape, dtype=torch.float64, device=s.x.device)
    for e in range(s.w1.shape[0]):
        for k in range(2):
            rows = (ids[:, k] == e).nonzero().reshape(-1)
            if rows.numel() == 0:
                continue
            x = s.x[rows].double()
            up = x @ s.w1[e].double().T
            up = up * torch.sigmoid(up) * (x @ s.w3[e].double().T)
            out[rows] += gates[rows, k, None] * (up @ s.w2[e].double().T)
    if hasattr(s, "moe_fn"):
        return {"out": out, "demand": demand}
    return {"out": out}


def _exact_attn(s):
    kv, seq = s.kv, s.kv.seq_len
    pos = torch.arange(seq, device=DEV)
    table = torch.tensor(kv.block_table, device=DEV)
    slots = table[pos // kv.block_size] * kv.block_size + pos % kv.block_size
    outs = []
    for layer, (q, k, v) in enumerate(s.qkv):
        n, hq, hd = q.shape
        group = hq // k.shape[1]
        keys = torch.cat([kv.k[layer].flatten(0, 1)[slots], k]).double()
        vals = torch.cat([kv.v[layer].flatten(0, 1)[slots], v]).double()
        keys = keys.permute(1, 2, 0).repeat_interleave(group, 0)         # [Hq, hd, S + N]
        vals = vals.permute(1, 0, 2).repeat_interleave(group, 0)         # [Hq, S + N, hd]
        score = torch.matmul(q.double().permute(1, 0, 2).contiguous(), keys.contiguous())
        score = score * hd ** -0.5
        score[:, :, seq:].masked_fill_(~s.mask[None], -math.inf)
        ctx = torch.matmul(torch.softmax(score, -1), vals.contiguous())  # [Hq, N, hd]
        outs.append(ctx.permute(1, 0, 2).reshape(n, hq * hd))
    return {"out": outs, "k": None, "v": None}


def exact(case, seed):
    """The computed numbers in 64 bits; op4 returns indices and copied bytes only."""
    if case["kind"] == "op4":
        return None
    s, kind = prepare(case, seed)
    return _exact_op1(s) if kind == "op1" else _exact_attn(s)
