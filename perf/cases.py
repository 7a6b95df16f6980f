"""The workloads this framework is measured on: one layer's (or one model's) sparse prefill through
the public entry points, from a single-head call on a short prompt to a 128K-token layer.

``listed()`` are the fixed cases, ``draw(rng)`` gives further ones of the same ranges; ``prepare``
makes a case's inputs on the GPU from a seed, ``run`` is one pass, ``work`` the bytes and operations
the pass cannot do without, ``tolerance`` how far another correct implementation may be off.

A case names its ``kind`` (the entry point), the token count ``n``, the head counts ``hq`` / ``hk``,
``d`` (head_dim), the ``dtype``, the ``batch`` and the memory ``layout`` of q/k/v: "bhnd" is a
contiguous [B, H, N, D] tensor, "bnhd" the transposed view of a projection's [B, N, H, D] output,
which is what a decoder layer hands over.
"""
import random

import torch

import minference_amd as M
from minference_amd.llama import LlamaConfig, LlamaPrefill

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, kind, n, hq=32, hk=8, d=128, dtype="bf16", batch=1, layout="bhnd", **more):
    c = {"kind": kind, "n": n, "hq": hq, "hk": hk, "d": d, "dtype": dtype, "batch": batch, "layout": layout, **more}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one head of a short prompt: the operator called head by head, as a per-head loop does
        _case("vs_head_4k", "vs", 4096, hq=1, hk=1, v=500, s=700),
        # a whole grouped-query layer of an ordinary prompt whose length is no multiple of anything
        _case("vs_layer_16k", "vs", 16001, v=1000, s=6096, layout="bnhd"),
        # a whole layer of a long prompt with the default pattern sizes: the headline workload
        _case("vs_layer_128k", "vs", 131072, v=1000, s=6096),
        # the operator on indices the caller selected (torch.topk order, int64), fp32 tensors
        _case("op_fp32_8k", "op", 8192, hq=4, hk=4, dtype="fp32", v=1000, s=2048),
        # a layer with a searched pattern table: all three pattern types and several sizes in one call
        _case("mixed_layer_50k", "mixed", 50000, layout="bnhd"),
        # the block-sparse operator: block index and attention, top-100
        _case("bs_layer_32k", "bs", 32768, top_k=100),
        # the sink + sliding window operator with the default sizes on a long ragged prompt
        _case("ashape_layer_100k", "ashape", 100000, n_init=128, n_local=3968, layout="bnhd"),
        # tri-shape on a model with 64-wide heads, no grouped queries, fp16
        _case("tri_fp16_d64_24k", "tri", 24000, hq=16, hk=16, d=64, dtype="fp16", n_init=8, n_local=512, n_last=128),
        # a layer below starting_layer: dense attention, two short prompts
        _case("dense_b2_6k", "dense", 6144, batch=2, layout="bnhd"),
        # the index builder alone with its full zero-filled outputs
        _case("index_256k", "index", 262144, hk=32, v=1000, s=6096),
        # the offline pattern search of one layer: all heads, all default candidates
        _case("search_16k", "search", 16384),
        # a decoder stack's prefill that keeps its K/V for decoding: two layers, default pattern
        _case("llama_2layers_32k", "llama", 32768, layers=2),
    ]


# smallest and largest token count that `draw` gives a kind
_RANGE = {"vs": (300, 131072), "op": (300, 32768), "mixed": (2000, 100000), "bs": (1000, 100000),
          "ashape": (500, 131072), "tri": (500, 65536), "dense": (300, 24000), "index": (4096, 262144),
          "search": (4096, 24000), "llama": (1000, 32768)}
_VS_SIZES = ((30, 800), (100, 750), (500, 700), (3500, 100), (1000, 6096))
_HEADS = ((1, 1), (4, 4), (8, 2), (16, 16), (28, 4), (32, 8), (32, 8))


def draw(rng):
    kind = rng.choice(sorted(_RANGE))
    lo, hi = _RANGE[kind]
    n = int(round(lo * (hi / lo) ** rng.random()))
    if rng.random() < 0.3:
        n = max(lo, n // 64 * 64)
    layout = rng.choice(("bhnd", "bnhd"))
    if kind == "llama":
        return _case(None, kind, n, layers=rng.choice((1, 2)))
    if kind == "index":
        hq = rng.choice((1, 4, 8, 16, 32))
        v, s = rng.choice(_VS_SIZES)
        return _case(None, kind, n, hq=hq, hk=hq, batch=rng.choice((1, 1, 2)) if n < 131072 else 1, v=v, s=s)
    hq, hk = rng.choice(_HEADS)
    d = rng.choice((128, 128, 128, 64)) if kind != "search" else 128
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    batch = rng.choice((1, 1, 1, 2)) if n <= 32768 else 1
    more = {}
    if kind in ("vs", "op"):
        more["v"], more["s"] = rng.choice(_VS_SIZES)
        if kind == "op" and n <= 8192 and rng.random() < 0.4:
            dtype = "fp32"
    elif kind == "mixed":
        hq, hk = rng.choice(((8, 2), (28, 4), (32, 8)))
        batch = 1
    elif kind == "bs":
        more["top_k"] = rng.choice((50, 100, 100))
    elif kind == "ashape":
        more["n_init"], more["n_local"] = rng.choice(((128, 3968), (128, 4096), (64, 1000), (4, 512)))
    elif kind == "tri":
        more["n_init"], more["n_local"], more["n_last"] = rng.choice(((8, 512, 128), (128, 3968, 100)))
    return _case(None, kind, n, hq=hq, hk=hk, d=d, dtype=dtype, batch=batch, layout=layout, **more)


# ---- inputs ---------------------------------------------------------------------------------------
def _store(x, layout):
    """x [B, H, N, D] in the case's memory layout (same shape, other strides)."""
    return x.transpose(1, 2).contiguous().transpose(1, 2) if layout == "bnhd" else x.contiguous()


def _qkv(case, seed):
    """Attention inputs with the structure long-context heads have: four sink keys, a few dozen heavy
    columns, a local band, and attention mass that halves every thousand tokens (an exact positional
    code in three of the head's dims adds a constant per token to a key's logit)."""
    B, hq, hk, n, d = case["batch"], case["hq"], case["hk"], case["n"], case["d"]
    dev, dt = torch.device("cuda"), _DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)
    group, sd = hq // hk, d ** 0.5
    a, gl, width = sd ** 0.5, (2.0 * sd) ** 0.5, min(512, n)
    q = torch.empty(B, hq, n, d, dtype=dt, device=dev)
    k = torch.empty(B, hk, n, d, dtype=dt, device=dev)
    v = torch.empty(B, hk, n, d, dtype=dt, device=dev)
    pos = torch.arange(n, device=dev)
    digits = torch.stack([pos // 16384, (pos // 128) % 128, pos % 128], 1).float()
    qconst = torch.tensor([128.0, 1.0, 2.0 ** -7], device=dev)
    for b in range(B):
        for j in range(hk):
            u = torch.randn(d, generator=g, device=dev)
            u[-3:] = 0
            u = u / u.norm()
            heavy = torch.randint(4, n, (32,), generator=g, device=dev)
            c = torch.cumsum(torch.randn(n, d, generator=g, device=dev, dtype=torch.float64), 0)
            z = c.clone()
            z[width:] -= c[:-width]
            z = (z / width ** 0.5).float() / sd                  # a smooth process: close rows are alike
            kk = torch.randn(n, d, generator=g, device=dev) + gl * z
            kk[:4] += (7.5 * sd / a) * u
            kk[heavy] += (4.0 * sd / a) * u
            kk[:, -3:] = digits
            k[b, j] = kk.to(dt)
            v[b, j] = torch.randn(n, d, generator=g, device=dev).to(dt)
            for i in range(group):
                qq = torch.randn(n, d, generator=g, device=dev) + gl * z + a * u
                qq[:, -3:] = qconst
                q[b, j * group + i] = qq.to(dt)
    return tuple(_store(x, case["layout"]) for x in (q, k, v))


def _distinct(rows, n, count, forced, tau, g):
    """`count` distinct numbers below n for each row, 0 .. forced-1 among them, in no particular
    order; with `tau` small numbers are the likelier ones (their odds fall by e every tau)."""
    dev = torch.device("cuda")
    u = torch.rand(rows, n, generator=g, device=dev)
    if tau:
        u = -torch.log(-torch.log(u.clamp(1e-7, 1 - 1e-7))) - torch.arange(n, device=dev) / tau
    u[:, :forced] += 1e9
    picked = torch.topk(u, min(count, n), dim=-1).indices
    return torch.gather(picked, 1, torch.rand(picked.shape, generator=g, device=dev).argsort(-1))


# one pattern table per head count, as a searched model has one for good
_TABLES = {}


def _table(hq):
    if hq not in _TABLES:
        rng, layer = random.Random(501), {}
        for h in range(hq):
            u = rng.random()
            if u < 0.7:
                v, s = rng.choice(_VS_SIZES + (_VS_SIZES[-1],) * 3)
                layer[str(h)] = ["vertical_and_slash", v, s, 1.0]
            elif u < 0.9:
                layer[str(h)] = ["block_sparse", 100, 0, 1.0]
            else:
                layer[str(h)] = ["stream_llm", 128, 4096, 1.0]
        _TABLES[hq] = [layer]
    return _TABLES[hq]


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    st = {"case": case}
    if kind == "llama":
        st["model"] = LlamaPrefill(LlamaConfig(num_layers=case["layers"]), seed=seed)
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        st["ids"] = torch.randint(0, 128256, (n,), generator=g, device="cuda")
        return st
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    B, H = case["batch"], case["hq"]
    if kind == "index":
        st["seqlens"] = torch.full((B,), n, dtype=torch.int32, device="cuda")
        st["v"] = _distinct(B * H, n, case["v"], 4, 0, g).sort(-1)[0].to(torch.int32).view(B, H, -1)
        st["s"] = _distinct(B * H, n, case["s"], 64, 0, g).sort(-1, descending=True)[0].to(torch.int32).view(B, H, -1)
        return st
    st["q"], st["k"], st["v"] = _qkv(case, seed)
    if kind == "op":
        st["v_idx"] = _distinct(B * H, n, case["v"], 30, 0, g).view(B, H, -1)
        st["s_idx"] = _distinct(B * H, n, case["s"], 100, n / 8, g).view(B, H, -1)
    elif kind == "mixed":
        st["kwargs"] = {"layer_idx": 0, "attn_forward_config": {"best_pattern": _table(H)}}
    return st


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "vs":
        return M.vertical_slash_prefill(st["q"], st["k"], st["v"], c["v"], c["s"])
    if kind == "op":
        return M.vertical_slash_sparse_attention(st["q"], st["k"], st["v"], st["v_idx"], st["s_idx"])
    if kind == "mixed":
        return M.minference_prefill_forward(st["q"], st["k"], st["v"], st["kwargs"])
    if kind == "bs":
        return M.block_sparse_attention(st["q"], st["k"], st["v"], c["top_k"])
    if kind == "ashape":
        return M.streaming_forward(st["q"], st["k"], st["v"], c["n_init"], c["n_local"])
    if kind == "tri":
        return M.tri_shape_forward(st["q"], st["k"], st["v"], c["n_init"], c["n_local"], c["n_last"])
    if kind == "dense":
        return M.dense_causal_attention(st["q"], st["k"], st["v"])
    if kind == "index":
        return M.convert_vertical_slash_indexes(st["seqlens"], st["v"], st["s"], c["n"])
    if kind == "search":
        return M.pattern_recall(st["q"], st["k"])
    if kind == "llama":
        return st["model"].prefill(st["ids"], keep_kv=True)
    raise KeyError(kind)


# ---- what a pass cannot do without ------------------------------------------------------------------
def _kept(n, most):
    """Sum over the query rows of the keys a row attends to when it keeps at most `most` of them."""
    m = min(n, most)
    return m * (m + 1) // 2 + (n - m) * m


def _layer_keys(case):
    """(query, key) pairs of one layer, all heads: the selected keys of every row, counted once."""
    n, kind = case["n"], case["kind"]
    heads = case["batch"] * case["hq"]
    if kind in ("vs", "op"):
        return heads * _kept(n, case["v"] + case["s"])
    if kind == "mixed":
        total = 0
        for ty, v, s, _ in _table(case["hq"])[0].values():
            total += _kept(n, 6400 if ty == "block_sparse" else v + s)
        return case["batch"] * total
    if kind == "bs":
        return heads * _kept(n, 64 * case["top_k"])
    if kind == "ashape":
        return heads * _kept(n, case["n_init"] + case["n_local"])
    if kind == "tri":
        last = min(case["n_last"], n)
        return heads * (_kept(n, case["n_init"] + case["n_local"]) + last * max(0, n - case["n_init"] - case["n_local"]))
    return heads * (n * (n + 1) // 2)                            # dense, search


def work(case):
    n, B, hq, hk, d = case["n"], case["batch"], case["hq"], case["hk"], case["d"]
    if case["kind"] == "index":
        rows = (n + 63) // 64
        v, s = min(case["v"], n), min(case["s"], n)
        return {"bytes": 4 * B * hq * (v + s + rows * (v + s + 2)), "flops": 0}
    size = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "llama":
        c, layers = LlamaConfig(), case["layers"]
        per_token = c.hidden_size * (c.num_heads + 2 * c.num_kv_heads) * c.head_dim \
            + c.num_heads * c.head_dim * c.hidden_size + 3 * c.hidden_size * c.intermediate_size
        keys = c.num_heads * _kept(n, 7096)
        kv = 2 * 2 * n * c.num_kv_heads * c.head_dim
        return {"bytes": layers * (2 * per_token + kv) + 2 * n * c.hidden_size + 2 * c.vocab_size * c.hidden_size,
                "flops": layers * (2 * n * per_token + 4 * c.head_dim * keys) + 2 * c.hidden_size * c.vocab_size}
    if case["kind"] == "search":
        return {"bytes": size * B * n * d * (hq + hk), "flops": 2 * d * _layer_keys(case)}
    return {"bytes": size * B * n * d * (2 * hq + 2 * hk), "flops": 4 * d * _layer_keys(case)}


def tolerance(case):
    """About four times what was measured: attention against an fp32 softmax 1.8e-3 (bf16), 2.3e-4
    (fp16), 6.6e-4 (fp32 tensors, computed on fp16 operands); index selections against fp64 scores
    rounded at the same points: the same sets; the search against an fp32 N x N softmax 2e-7, where a
    tie in its top-k may weigh more; the decoder stack against itself with norms or rotary embedding in
    fp64 7.6e-3 (logits) and 4.7e-3 (K/V of the second layer)."""
    kind = case["kind"]
    if kind == "index":
        return "exact"
    if kind == "search":
        return {"rel": 1e-5}
    if kind == "llama":
        return {"rel": 3e-2}
    return {"rel": {"bf16": 8e-3, "fp16": 1e-3, "fp32": 2.5e-3}[case["dtype"]]}
