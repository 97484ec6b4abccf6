"""Performance cases of the packed target-verification path.

Each case is one call (or one small group of calls that always follow each
other) of the public entry points, on inputs like those a verification wave
has: packed tree attention, the KV commit, tree sampling, the LM head with
its walk, the fused stages of a decoder layer, and one whole decoder stack.

  attn    ops.tree_attention over one wave (a layer's call; the wave's plan is
          made once and shared by all layers, so it is part of the state)
  sample  ops.tree_sample over every row's logits
  lazy    ops.lm_head over the internal rows, then ops.tree_sample_projected
  head    ops.lm_head alone (the reached leaves, or a few rows)
  layer   target.add_rmsnorm, qk_norm_rope, add_rmsnorm, silu_mul of one layer
  commit  ops.kv_commit of every layer's accepted rows
  stack   attention mask, plan, Qwen3TargetStack forward and logits of a wave
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

from specgrove_amd import attention, cache, ops, target
from specgrove_amd import workloads as W

BF16 = torch.bfloat16
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DEVICE = "cuda:0"


def listed():
    return [
        # Smallest call: a 2-layer test-size model's wave, four 16-node trees.
        {"name": "attn_tiny", "kind": "attn", "requests": 4, "prefix_lo": 32, "prefix_hi": 96,
         "tiers": "16", "budget": 64, "hq": 4, "hkv": 2, "dim": 64, "tree": "random", "wave": 1},
        # A lightly loaded server: 16 requests, short contexts, 512-row budget.
        {"name": "attn_16req", "kind": "attn", "requests": 16, "prefix_lo": 256,
         "prefix_hi": 2048, "tiers": "16,32,64", "budget": 512, "hq": 32, "hkv": 8, "dim": 128,
         "tree": "canonical", "wave": 2},
        # The ordinary wave: 64 requests, 2048-row budget.
        {"name": "attn_64req", "kind": "attn", "requests": 64, "prefix_lo": 512,
         "prefix_hi": 4096, "tiers": "16,32,64,128", "budget": 2048, "hq": 32, "hkv": 8,
         "dim": 128, "tree": "canonical", "wave": 3},
        # Prefill: chunks of 256 prompt tokens (causal chains) of eight prompts.
        {"name": "attn_prefill", "kind": "attn", "requests": 8, "prefix_lo": 256,
         "prefix_hi": 3072, "tiers": "256", "budget": 2048, "hq": 32, "hkv": 8, "dim": 128,
         "tree": "chain", "wave": 4},
        # The largest wave: 128 requests with 8k to 32k cached tokens.
        {"name": "attn_long", "kind": "attn", "requests": 128, "prefix_lo": 8192,
         "prefix_hi": 32768, "tiers": "1,16,32,64,128", "budget": 4096, "hq": 32, "hkv": 8,
         "dim": 128, "tree": "canonical", "wave": 5},
        # Verification of a full wave from fp32 logits.
        {"name": "sample_f32", "kind": "sample", "requests": 64, "nodes_lo": 32, "nodes_hi": 32,
         "vocab": 151936, "dtype": "f32", "wave": 6},
        # Ragged trees and a vocabulary that is not a multiple of the vector width.
        {"name": "sample_bf16_odd", "kind": "sample", "requests": 24, "nodes_lo": 1,
         "nodes_hi": 64, "vocab": 50257, "dtype": "bf16", "wave": 7},
        # Lazy verification: internal rows of an ordinary wave, packed head weight.
        {"name": "lazy_64req", "kind": "lazy", "requests": 64, "nodes_lo": 16, "nodes_hi": 48,
         "hidden": 4096, "vocab": 151936, "packed": True, "wave": 8},
        # Its second pass: one reached leaf per request.
        {"name": "head_leaves", "kind": "head", "rows": 64, "hidden": 4096, "vocab": 151936,
         "packed": True, "wave": 9},
        # The fused stages of one decoder layer over an ordinary wave.
        {"name": "layer_stages", "kind": "layer", "rows": 2048, "hidden": 4096,
         "intermediate": 12288, "hq": 32, "hkv": 8, "dim": 128, "wave": 10},
        # The accepted rows of a wave into the cache arena of 36 layers.
        {"name": "commit_36", "kind": "commit", "requests": 64, "layers": 36, "hkv": 8,
         "dim": 128, "rows": 32, "keep_hi": 9, "wave": 11},
        # A whole target call of a lightly loaded server, four layers of it.
        {"name": "stack_16req", "kind": "stack", "requests": 16, "prefix_lo": 256,
         "prefix_hi": 2048, "tiers": "16,32,64", "budget": 512, "hq": 32, "hkv": 8, "dim": 128,
         "tree": "canonical", "layers": 4, "hidden": 2560, "intermediate": 9728,
         "vocab": 151936, "wave": 12},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges above, odd sizes among them."""
    kind = rng.choices(["attn", "sample", "lazy", "head", "layer", "commit"],
                       [8, 4, 2, 3, 2, 1])[0]
    wave = rng.randrange(1 << 30)
    if kind == "attn":
        tree = rng.choice(["canonical", "canonical", "random", "chain"])
        tiers = rng.choice(["1,16,32,64,128", "16,32,64", "16,32,64,128", "32", "128"]
                           if tree != "chain" else ["1,7,64,200,256", "256", "1"])
        requests = min(_log_int(rng, 2, 128), 4096 // int(tiers.split(",")[0]))
        budget = min(4096, 128 * requests if tree != "chain" else 256 * requests)
        hq, hkv = rng.choice([(32, 8), (32, 8), (4, 2), (16, 8), (64, 8), (16, 16), (32, 2)])
        hi = _log_int(rng, 64, min(32768, 2300000 // requests, 2500000000 // (budget * hq)))
        lo = max(1, int(hi / rng.choice([1.0, 2.0, 4.0, 8.0])))
        return {"kind": kind, "requests": requests, "prefix_lo": lo, "prefix_hi": hi,
                "tiers": tiers, "budget": budget, "hq": hq, "hkv": hkv,
                "dim": rng.choice([64, 128, 128]), "tree": tree, "wave": wave}
    if kind == "sample":
        hi = _log_int(rng, 4, 64)
        return {"kind": kind, "requests": _log_int(rng, 2, 1024 // max(hi, 16)),
                "nodes_lo": rng.choice([1, hi // 2, hi]), "nodes_hi": hi,
                "vocab": rng.choice([151936, _log_int(rng, 8000, 151936),
                                     4 * _log_int(rng, 2000, 37984)]),
                "dtype": rng.choice(["f32", "bf16", "bf16", "f16"]), "wave": wave}
    if kind == "lazy":
        hi = _log_int(rng, 4, 48)
        return {"kind": kind, "requests": _log_int(rng, 2, 48), "nodes_lo": max(2, hi // 3),
                "nodes_hi": hi, "hidden": rng.choice([512, 2560, 4096]),
                "vocab": rng.choice([151936, _log_int(rng, 8000, 151936)]),
                "packed": rng.random() < 0.6, "wave": wave}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 2, 640),
                "hidden": rng.choice([512, 1024, 2560, 4096]),
                "vocab": rng.choice([151936, _log_int(rng, 8000, 151936)]),
                "packed": rng.random() < 0.6, "wave": wave}
    if kind == "layer":
        hidden, inter, hq, hkv, dim = rng.choice(
            [(4096, 12288, 32, 8, 128), (2560, 9728, 32, 8, 128), (256, 768, 4, 2, 64)])
        return {"kind": kind, "rows": _log_int(rng, 16, 4096), "hidden": hidden,
                "intermediate": inter, "hq": hq, "hkv": hkv, "dim": dim, "wave": wave}
    return {"kind": "commit", "requests": _log_int(rng, 2, 64), "layers": rng.choice([1, 2, 36]),
            "hkv": rng.choice([2, 8]), "dim": rng.choice([64, 128]), "rows": rng.choice([9, 32]),
            "keep_hi": rng.choice([2, 9]), "wave": wave}


# --------------------------------------------------------------------------
# shapes of a case (from its values alone)
# --------------------------------------------------------------------------

def _tree(kind, nodes, nprng):
    if kind == "chain":
        return [-1] + list(range(nodes - 1))
    if kind == "random":
        return W.random_parent_tree(nodes, nprng, max_depth=16)
    return W.canonical_tree(nodes, nprng)


def _attention_wave(c):
    rng = np.random.default_rng(c["wave"])
    options = [int(t) for t in c["tiers"].split(",")]
    n = c["requests"]
    lengths = np.floor(np.exp(rng.uniform(math.log(c["prefix_lo"]),
                                          math.log(c["prefix_hi"] + 1), n))).astype(np.int32) \
        if c["prefix_hi"] > 4096 else \
        rng.integers(c["prefix_lo"], c["prefix_hi"] + 1, n).astype(np.int32)
    tiers = [int(t) for t in rng.choice(options, size=n)]
    if sum(tiers) > c["budget"] and options[0] * n <= c["budget"]:
        tiers = W.downgrade_tiers(tiers, options, c["budget"])
    full = _tree(c["tree"], max(options), rng)
    parents = [full[:t] for t in tiers]
    capacity = (int(lengths.max()) + max(options) + 9 + 63) // 64 * 64
    return W.AttentionWorkload("wave", c["hq"], c["hkv"], c["dim"], lengths, parents,
                               [[0] * (t - 1) for t in tiers], capacity)


def _trees(c):
    """Parents of the sampled trees, and each node's rank among its siblings."""
    rng = np.random.default_rng(c["wave"])
    sizes = rng.integers(c["nodes_lo"], c["nodes_hi"] + 1, c["requests"])
    parents = [W.canonical_tree(int(s), rng) for s in sizes]
    ranks = []
    for p in parents:
        seen = {}
        for v in p:
            ranks.append(seen.get(v, 0))
            seen[v] = ranks[-1] + 1
    return parents, np.asarray(ranks, np.int64)


def _pack(parents):
    offset = np.concatenate([[0], np.cumsum([len(p) for p in parents])]).astype(np.int32)
    parent = np.concatenate([np.asarray(p, np.int32) for p in parents])
    owner = np.repeat(np.arange(len(parents)), np.diff(offset))
    packed_parent = np.where(parent >= 0, parent + offset[owner], -1).astype(np.int64)
    return offset, parent, packed_parent


def _depth(parents):
    return max(max(W.depths_of(p)) for p in parents)


def _internal(parents):
    _, _, packed_parent = _pack(parents)
    return np.unique(packed_parent[packed_parent >= 0]).astype(np.int32)


def _keep_lens(c):
    rng = np.random.default_rng(c["wave"])
    return rng.integers(1, min(c["keep_hi"], c["rows"]) + 1, c["requests"]).astype(np.int32)


def work(c):
    kind = c["kind"]
    if kind == "attn":
        wl = _attention_wave(c)
        return {"bytes": wl.algorithmic_bytes(), "flops": wl.algorithmic_flops()}
    if kind == "sample":
        rows = sum(len(p) for p in _trees(c)[0])
        size = 4 if c["dtype"] == "f32" else 2
        return {"bytes": rows * c["vocab"] * size, "flops": 0}
    if kind in ("lazy", "head"):
        rows = c["rows"] if kind == "head" else len(_internal(_trees(c)[0]))
        h, v = c["hidden"], c["vocab"]
        return {"bytes": 2 * (v * h + rows * h + rows * v), "flops": 2 * rows * h * v}
    if kind == "layer":
        qkv = (c["hq"] + 2 * c["hkv"]) * c["dim"]
        per_row = 2 * 4 * c["hidden"] + 2 * qkv + 3 * c["intermediate"]
        return {"bytes": 2 * c["rows"] * per_row, "flops": 0}
    if kind == "commit":
        rows = int(_keep_lens(c).sum())
        return {"bytes": 2 * rows * c["hkv"] * c["dim"] * 2 * 2 * c["layers"], "flops": 0}
    wl = _attention_wave(c)
    h, i, v, r = c["hidden"], c["intermediate"], c["vocab"], wl.total_rows
    weights = c["layers"] * (h * (c["hq"] + 2 * c["hkv"]) * c["dim"] + c["hq"] * c["dim"] * h
                             + 3 * h * i) + v * h
    return {"bytes": 2 * (weights + r * v) + c["layers"] * wl.algorithmic_bytes(),
            "flops": 2 * r * weights + c["layers"] * wl.algorithmic_flops()}


def tolerance(c):
    """Copies and the sampler's fixed-order fp32 arithmetic are exact.  The
    others: about four times the distance from the result in 64 bits (bf16
    operands or results; a few roundings in a row for the layer's stages and
    the stack), for the head's logits twice their own rounding."""
    return {"attn": {"rel": 1e-2, "max": 0.2},
            "sample": "exact",
            "lazy": {"rel": 4e-3, "max": 0.1, "differ": 0.005},
            "head": {"rel": 4e-3, "max": 0.1},
            "layer": {"rel": 1e-2, "max": 0.1},
            "commit": "exact",
            "stack": {"rel": 3e-2, "max": 0.5}}[c["kind"]]


# --------------------------------------------------------------------------
# states
# --------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(g, *shape, scale=1.0, dtype=BF16):
    t = torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)
    return t.mul_(scale) if scale != 1.0 else t


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)


def _prepare_attn(c, seed):
    wl = _attention_wave(c)
    q, kc, vc, kt, vt = wl.make_tensors(DEVICE, seed, q_scale=1.5)
    plan = ops.plan_attention(wl.row_offset, wl.prefix_len, wl.num_q_heads, wl.num_kv_heads,
                              wl.head_dim).to(DEVICE)
    return {"args": (q, kc, vc, kt, vt, _dev(wl.row_offset), _dev(wl.prefix_start),
                     _dev(wl.prefix_len), _dev(wl.parent_flat), plan)}


def _logit_rows(g, rows, vocab, dtype):
    """Logits of a language model's spread, with one to five likely tokens a row."""
    logits = _randn(g, rows, vocab, scale=3.0, dtype=torch.float32)
    for _ in range(5):
        col = torch.randint(0, vocab, (rows, 1), generator=g, device=DEVICE)
        on = (torch.rand((rows, 1), generator=g, device=DEVICE) < 0.6).float() * 12.0
        logits.scatter_add_(1, col, on)
    return logits.to(dtype)


def _prepare_sample(c, seed):
    g = _gen(seed)
    parents, ranks = _trees(c)
    offset, parent, packed_parent = _pack(parents)
    rows = len(parent)
    logits = _logit_rows(g, rows, c["vocab"], DTYPES[c["dtype"]])
    # Draft children: distinct tokens among the target row's likeliest sixteen.
    top = logits.float().topk(16, dim=1).indices
    order = torch.rand((rows, 16), generator=g, device=DEVICE).argsort(1)
    token = top.gather(1, order)[_dev(np.maximum(packed_parent, 0)), _dev(ranks)]
    token = torch.where(_dev(packed_parent) >= 0, token, 0).to(torch.int32)
    depth = _depth(parents)
    uniforms = torch.rand((len(parents), 2 * (depth + 1)), generator=g, device=DEVICE)
    return {"args": (logits, _dev(offset), _dev(parent), token.contiguous(), uniforms, depth)}


def _head_weight(g, vocab, hidden, packed):
    weight = _randn(g, vocab, hidden, scale=3.0 / math.sqrt(hidden))
    return weight, (ops.pack_lm_head(weight) if packed else weight)


def _prepare_head(c, seed):
    g = _gen(seed)
    total = 2 * c["rows"] + 1
    weight, head = _head_weight(g, c["vocab"], c["hidden"], c["packed"])
    hidden = _randn(g, total, c["hidden"])
    index = torch.randperm(total, generator=g, device=DEVICE)[:c["rows"]].to(torch.int32)
    return {"hidden": hidden, "head": head, "index": index, "weight": weight}


def _prepare_lazy(c, seed):
    g = _gen(seed)
    parents, ranks = _trees(c)
    offset, parent, packed_parent = _pack(parents)
    rows, internal = len(parent), _internal(parents)
    weight, head = _head_weight(g, c["vocab"], c["hidden"], c["packed"])
    # Distinct draft tokens, each likely in its parent's row (the parent's
    # hidden state leans towards the token's head row).
    token = torch.randperm(c["vocab"], generator=g, device=DEVICE)[
        torch.arange(rows, device=DEVICE) % c["vocab"]]
    hidden = _randn(g, rows, c["hidden"], dtype=torch.float32)
    lean = weight[token].float()
    lean = lean * (14.0 / lean.square().sum(1, keepdim=True))
    edge = _dev(packed_parent) >= 0
    for rank in range(int(ranks.max()) + 1):  # one child of each parent at a time
        on = np.flatnonzero((packed_parent >= 0) & (ranks == rank))
        hidden[_dev(packed_parent[on])] += lean[_dev(on)]
    token = torch.where(edge, token, -1).to(torch.int32)
    row_map = np.full(rows, -1, np.int32)
    row_map[internal] = np.arange(len(internal), dtype=np.int32)
    depth = _depth(parents)
    uniforms = torch.rand((len(parents), 2 * (depth + 1)), generator=g, device=DEVICE)
    return {"hidden": hidden.to(BF16), "head": head, "index": _dev(internal), "weight": weight,
            "walk": (_dev(offset), _dev(parent), token, uniforms, depth),
            "row_map": _dev(row_map)}


def _inv_freq(dim):
    return (1.0 / (1e6 ** (torch.arange(0, dim, 2, dtype=torch.int64).float() / dim))).to(DEVICE)


def _norm_weight(g, n):
    return (1.0 + _randn(g, n, scale=0.1, dtype=torch.float32)).to(BF16)


def _prepare_layer(c, seed):
    g = _gen(seed)
    r, h, d = c["rows"], c["hidden"], c["dim"]
    return {"case": c,
            "x1": _randn(g, r, h), "res1": _randn(g, r, h, scale=2.0), "w1": _norm_weight(g, h),
            "qkv": _randn(g, r, (c["hq"] + 2 * c["hkv"]) * d),
            "qn": _norm_weight(g, d), "kn": _norm_weight(g, d), "inv_freq": _inv_freq(d),
            "pos": torch.randint(0, 32768, (r,), generator=g, device=DEVICE),
            "x2": _randn(g, r, h), "res2": _randn(g, r, h, scale=2.0), "w2": _norm_weight(g, h),
            "gate_up": _randn(g, r, 2 * c["intermediate"])}


def _prepare_commit(c, seed):
    g = _gen(seed)
    n, layers, hkv, d, rows = c["requests"], c["layers"], c["hkv"], c["dim"], c["rows"]
    rng = np.random.default_rng(seed)
    keep_len = _keep_lens(c)
    stride = int(keep_len.max())
    keep = np.full((n, stride), -1, np.int32)
    for i, k in enumerate(keep_len):
        keep[i, 0] = 0
        keep[i, 1:k] = 1 + np.sort(rng.permutation(rows - 1)[:k - 1])
    capacity = 160
    arena = _randn(g, 2, layers, hkv, n * capacity, d)
    tree = _randn(g, 2, layers, n * rows, hkv, d)
    pointers = [ops.pointer_array(list(t.unbind(0)), DEVICE) for t in (*arena, *tree)]
    lengths = rng.integers(64, 145, n).astype(np.int32)
    return {"arena": arena, "tree": tree, "pointers": pointers, "base": _dev(lengths),
            "lengths": _dev(lengths),
            "kw": dict(num_kv_heads=hkv, head_dim=d, cache_head_stride=arena.stride(2),
                       cache_token_stride=arena.stride(3), tree_row_stride=tree.stride(2),
                       tree_head_stride=tree.stride(3),
                       row_offset=_dev(np.arange(n + 1, dtype=np.int32) * rows),
                       keep_rows=_dev(keep), keep_len=_dev(keep_len),
                       prefix_start=_dev(np.arange(n, dtype=np.int64) * capacity),
                       capacity=capacity)}


def _prepare_stack(c, seed):
    g = _gen(seed)
    wl = _attention_wave(c)
    h, i, d, hq, hkv = c["hidden"], c["intermediate"], c["dim"], c["hq"], c["hkv"]

    def linear(out, inp, bias=None):
        return SimpleNamespace(weight=_randn(g, out, inp, scale=1.0 / math.sqrt(inp)), bias=bias)

    def norm(n):
        return SimpleNamespace(weight=_norm_weight(g, n))

    layers = [SimpleNamespace(
        self_attn=SimpleNamespace(q_proj=linear(hq * d, h), k_proj=linear(hkv * d, h),
                                  v_proj=linear(hkv * d, h), o_proj=linear(h, hq * d),
                                  q_norm=norm(d), k_norm=norm(d)),
        mlp=SimpleNamespace(gate_proj=linear(i, h), up_proj=linear(i, h), down_proj=linear(h, i)),
        input_layernorm=norm(h), post_attention_layernorm=norm(h)) for _ in range(c["layers"])]
    model = SimpleNamespace(
        config=SimpleNamespace(model_type="qwen3", rope_theta=1e6, num_attention_heads=hq,
                               num_key_value_heads=hkv, head_dim=d, rms_norm_eps=1e-6),
        model=SimpleNamespace(layers=layers, norm=norm(h), embed_tokens=SimpleNamespace(
            weight=_randn(g, c["vocab"], h))),
        lm_head=SimpleNamespace(weight=_randn(g, c["vocab"], h, scale=3.0 / math.sqrt(h))))
    caches = []
    for length in wl.prefix_len:
        one = cache.RequestCache()
        for layer in range(c["layers"]):
            one.update(_randn(g, 1, hkv, int(length), d), _randn(g, 1, hkv, int(length), d),
                       layer)
        caches.append(one)
    pool = cache.PersistentRequestCachePool(caches, wl.capacity)
    depths = np.concatenate([np.asarray(W.depths_of(p)) for p in wl.parents])
    positions = depths + np.repeat(wl.prefix_len, wl.rows)
    ids = torch.randint(0, c["vocab"], (1, wl.total_rows), generator=g, device=DEVICE)
    return {"stack": target.Qwen3TargetStack.from_transformers(model), "pool": pool, "ids": ids,
            "parents": wl.parents, "positions": _dev(positions.astype(np.int64))[None]}


def prepare(case, seed):
    return {"kind": case["kind"], **{
        "attn": _prepare_attn, "sample": _prepare_sample, "lazy": _prepare_lazy,
        "head": _prepare_head, "layer": _prepare_layer, "commit": _prepare_commit,
        "stack": _prepare_stack}[case["kind"]](case, seed)}


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "attn":
        return ops.tree_attention(*s["args"])
    if kind == "sample":
        r = ops.tree_sample(*s["args"])
        return {"accept_nodes": r.accept_nodes, "accept_len": r.accept_len, "bonus": r.bonus,
                "keep_rows": r.keep_rows, "row_max": r.row_max, "row_sum": r.row_sum}
    if kind in ("head", "lazy"):
        head = ops.lm_head(s["hidden"], s["head"], s["index"])
        out = {"logits": head.logits, "row_max": head.row_max, "row_sum": head.row_sum}
        if kind == "lazy":
            r = ops.tree_sample_projected(head.logits, *s["walk"], row_max=head.row_max,
                                          row_sum=head.row_sum, row_map=s["row_map"])
            out.update(accept_nodes=r.accept_nodes, accept_len=r.accept_len, bonus=r.bonus,
                       keep_rows=r.keep_rows, terminal_leaf=r.terminal_leaf)
        return out
    if kind == "layer":
        c = s["case"]
        h1, sum1 = target.add_rmsnorm(s["x1"], s["w1"], 1e-6, s["res1"], want_sum=True)
        q, k, v = target.qk_norm_rope(s["qkv"], c["hq"], c["hkv"], c["dim"], s["qn"], s["kn"],
                                      s["inv_freq"], s["pos"], 1e-6)
        h2, sum2 = target.add_rmsnorm(s["x2"], s["w2"], 1e-6, s["res2"], want_sum=True)
        act = target.silu_mul(s["gate_up"])
        return {"h1": h1, "sum1": sum1, "q": q, "k": k, "v": v, "h2": h2, "sum2": sum2,
                "act": act}
    if kind == "commit":
        # A wave brings its requests' current lengths along.
        s["lengths"].copy_(s["base"])
        ops.kv_commit(*s["pointers"], lengths=s["lengths"], **s["kw"])
        return {"arena": s["arena"], "lengths": s["lengths"]}
    pool, stack = s["pool"], s["stack"]
    wave = cache.TreeVerifyCache(pool, pool.caches)
    mask = attention.build_tree_mask(pool, pool.caches, s["parents"], DEVICE)
    hidden = stack.model(input_ids=s["ids"], position_ids=s["positions"],
                         attention_mask={"full_attention": mask}, past_key_values=wave,
                         use_cache=True).last_hidden_state
    return {"hidden": hidden, "logits": stack.get_output_embeddings()(hidden),
            "keys": [layer.keys for layer in wave.layers],
            "values": [layer.values for layer in wave.layers]}


# --------------------------------------------------------------------------
# the same results in 64 bits
# --------------------------------------------------------------------------

def _attend(wl, q, kc, vc, kt, vt):
    """Tree attention of a wave, q [R, Hq, D], caches [Hkv, T, D], rows [R, Hkv, D]."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    group, d = wl.num_q_heads // wl.num_kv_heads, wl.head_dim
    for i, parents in enumerate(wl.parents):
        n, length = len(parents), int(wl.prefix_len[i])
        r0, p0 = int(wl.row_offset[i]), int(wl.prefix_start[i])
        seen = np.eye(n, dtype=bool)
        for k in range(1, n):
            seen[k] |= seen[parents[k]]
        hidden = ~_dev(seen).repeat_interleave(group, 0)
        for g in range(wl.num_kv_heads):
            keys = torch.cat([kc[g, p0:p0 + length], kt[r0:r0 + n, g]]).double()
            values = torch.cat([vc[g, p0:p0 + length], vt[r0:r0 + n, g]]).double()
            heads = slice(g * group, (g + 1) * group)
            scores = q[r0:r0 + n, heads].reshape(n * group, d).double() @ keys.t().contiguous()
            scores.mul_(d ** -0.5)[:, length:].masked_fill_(hidden, -math.inf)
            out[r0:r0 + n, heads] = (torch.softmax(scores, 1) @ values).view(n, group, d)
    return out


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, inv_freq):
    """x [R, heads, D] rotated (rotate-half form)."""
    angle = pos.double()[:, None] * inv_freq.double()
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _heads(qkv, c):
    hq, hkv, d = c["hq"], c["hkv"], c["dim"]
    rows = qkv.shape[0]
    return (qkv[:, :hq * d].reshape(rows, hq, d),
            qkv[:, hq * d:(hq + hkv) * d].reshape(rows, hkv, d),
            qkv[:, (hq + hkv) * d:].reshape(rows, hkv, d))


def _row_sums(x):
    m = x.max(1).values
    return m, torch.exp(x - m[:, None]).sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "commit":
        return None
    s = prepare(case, seed)
    if kind == "attn":
        return _attend(_attention_wave(case), *s["args"][:5])
    if kind == "sample":
        sums = [_row_sums(rows.double()) for rows in s["args"][0].split(256)]
        return {"row_max": torch.cat([m for m, _ in sums]),
                "row_sum": torch.cat([z for _, z in sums]),
                "accept_nodes": None, "accept_len": None, "bonus": None, "keep_rows": None}
    if kind in ("head", "lazy"):
        rows = s["hidden"][s["index"].long()].double()
        logits = torch.cat([rows @ w.double().t().contiguous()
                            for w in s["weight"].split(16384)], 1)
        m, z = _row_sums(logits)
        return {"logits": logits, "row_max": m, "row_sum": z}
    if kind == "layer":
        sums = [s["x1"].double() + s["res1"].double(), s["x2"].double() + s["res2"].double()]
        q, k, v = _heads(s["qkv"].double(), case)
        gate, up = s["gate_up"].double().chunk(2, 1)
        q = _rope(_rms(q, s["qn"]), s["pos"], s["inv_freq"])
        k = _rope(_rms(k, s["kn"]), s["pos"], s["inv_freq"])
        return {"h1": _rms(sums[0], s["w1"]), "sum1": sums[0], "h2": _rms(sums[1], s["w2"]),
                "sum2": sums[1], "q": q, "k": k.transpose(0, 1), "v": v.transpose(0, 1),
                "act": gate * torch.sigmoid(gate) * up}
    wl, stack, pool = _attention_wave(case), s["stack"], s["pool"]
    x = stack.embed[s["ids"][0]].double()
    pos = s["positions"][0]
    keys, values = [], []
    for index, layer in enumerate(stack.layers):
        q, k, v = _heads(_rms(x, layer.ln1) @ layer.wqkv.double().t(), case)
        q = _rope(_rms(q, layer.q_norm), pos, stack.inv_freq)
        k = _rope(_rms(k, layer.k_norm), pos, stack.inv_freq)
        keys.append(k.transpose(0, 1)[None])
        values.append(v.transpose(0, 1)[None])
        attended = _attend(wl, q, pool.key_storage[index], pool.value_storage[index], k, v)
        x = x + attended.reshape(x.shape[0], -1) @ layer.wo.double().t()
        gate, up = (_rms(x, layer.ln2) @ layer.wgu.double().t()).chunk(2, 1)
        x = x + (gate * torch.sigmoid(gate) * up) @ layer.wd.double().t()
    hidden = _rms(x, stack.norm)
    return {"hidden": hidden[None], "logits": (hidden @ stack.lm_head.weight.double().t())[None],
            "keys": keys, "values": values}
