"""Long-context prefill of a Llama-architecture decoder around the sparse attention path.

A caller of the path, not part of it: the counterpart of the reference's Llama patch
(minference/patch.py:688-693 chunked MLP, :500-558 chunked norms, :787-790 last-token lm_head;
minference/modules/forward.py:22-234 attention forward that hands [B,H,N,D] q/k/v to
``prefill_forwards["minference"]``) as a self-contained block stack instead of a monkey patch of
a particular transformers version.  Linear layers are plain library GEMMs (torch matmul ->
hipBLASLt); everything between the q/k/v projections and o_proj is
``minference_prefill_forward``; norms (with the residual add before them), rotary embedding and
SiLU * up are one kernel each (csrc/decoder.hip).  K/V keep their own (fewer) heads: no repeat_kv copy.

Memory layout for 262144 tokens of Llama-3-8B on one 288 GB GPU: weights 16 GB, hidden state and its
norm 2 GiB each, q and the attention output 2 GiB each, k/v 0.5 GiB each per layer; projections and
the MLP are applied over token chunks so no intermediate is larger than ``chunk x intermediate_size``.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from . import _lib
from .prefill import minference_prefill_forward


@dataclass
class LlamaConfig:
    """Defaults are Llama-3-8B."""
    vocab_size: int = 128256
    hidden_size: int = 4096
    intermediate_size: int = 14336
    num_layers: int = 32
    num_heads: int = 32
    num_kv_heads: int = 8
    head_dim: int = 128
    rope_theta: float = 500000.0
    rms_eps: float = 1e-5


class LlamaPrefill:
    """Random-init (or caller-filled) decoder weights + a chunked prefill that returns the
    last token's logits.  Weight names follow the Hugging Face Llama state dict."""

    def __init__(self, config: LlamaConfig, device="cuda", dtype=torch.bfloat16, seed=0, std=0.02):
        self.cfg, self.device, self.dtype = config, torch.device(device), dtype
        self._dt = {torch.bfloat16: _lib.MINF_BF16, torch.float16: _lib.MINF_F16, torch.float32: _lib.MINF_F32}.get(dtype)
        c = config
        g = torch.Generator(device=self.device).manual_seed(seed)

        def w(*shape):
            return (torch.randn(*shape, device=self.device, dtype=torch.float32, generator=g) * std).to(dtype)

        qd, kd = c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim
        self.embed_tokens = w(c.vocab_size, c.hidden_size)
        self.layers = []
        for _ in range(c.num_layers):
            self.layers.append({
                "input_layernorm": torch.ones(c.hidden_size, device=self.device, dtype=dtype),
                "q_proj": w(qd, c.hidden_size), "k_proj": w(kd, c.hidden_size), "v_proj": w(kd, c.hidden_size),
                "o_proj": w(c.hidden_size, qd),
                "post_attention_layernorm": torch.ones(c.hidden_size, device=self.device, dtype=dtype),
                "gate_proj": w(c.intermediate_size, c.hidden_size), "up_proj": w(c.intermediate_size, c.hidden_size),
                "down_proj": w(c.hidden_size, c.intermediate_size),
            })
        self.norm = torch.ones(c.hidden_size, device=self.device, dtype=dtype)
        self.lm_head = w(c.vocab_size, c.hidden_size)

    def load_state_dict(self, sd):
        """Fill the weights from a Hugging Face Llama state dict (tensors are cast and moved)."""
        def get(name):
            return sd[name].to(self.device, self.dtype)
        self.embed_tokens = get("model.embed_tokens.weight")
        for i, layer in enumerate(self.layers):
            pre = f"model.layers.{i}."
            for k in ("input_layernorm", "post_attention_layernorm"):
                layer[k] = get(pre + k + ".weight")
            for k in ("q_proj", "k_proj", "v_proj", "o_proj"):
                layer[k] = get(pre + "self_attn." + k + ".weight")
            for k in ("gate_proj", "up_proj", "down_proj"):
                layer[k] = get(pre + "mlp." + k + ".weight")
        self.norm = get("model.norm.weight")
        self.lm_head = get("lm_head.weight") if "lm_head.weight" in sd else self.embed_tokens

    # ---- pieces ---------------------------------------------------------------------------
    def _rms(self, x, weight, delta=None, out=None):
        """RMSNorm of the rows of x (contiguous); with ``delta`` x += delta first, in place."""
        out = torch.empty_like(x) if out is None else out
        lib = _lib.load()
        with torch.cuda.device(x.device):
            st = lib.minf_rms_norm(x.data_ptr(), delta.data_ptr() if delta is not None else None, weight.data_ptr(),
                                   out.data_ptr(), x.shape[0], x.shape[1], self.cfg.rms_eps, self._dt, _lib.stream_ptr(x.device))
        _lib.check(st, "minf_rms_norm")
        return out

    def _rope_tables(self, n):
        """cos, sin [n, D/2] fp32 (rotate_half convention: pairs (i, i + D/2) share an angle)."""
        c = self.cfg
        inv = 1.0 / (c.rope_theta ** (torch.arange(0, c.head_dim, 2, device=self.device, dtype=torch.float32) / c.head_dim))
        ang = torch.arange(n, device=self.device, dtype=torch.float32)[:, None] * inv[None, :]
        return ang.cos(), ang.sin()

    def _rotate(self, q, k, cos, sin):
        """Rotary embedding of q [n, Hq, D] and k [n, Hk, D] in place."""
        lib = _lib.load()
        with torch.cuda.device(q.device):
            st = lib.minf_rope(q.data_ptr(), k.data_ptr(), cos.data_ptr(), sin.data_ptr(), q.shape[0], q.shape[1],
                               k.shape[1], q.shape[2], self._dt, _lib.stream_ptr(q.device))
        _lib.check(st, "minf_rope")

    def _silu_mul(self, gate, up):
        """gate <- silu(gate) * up."""
        lib = _lib.load()
        with torch.cuda.device(gate.device):
            st = lib.minf_silu_mul(gate.data_ptr(), up.data_ptr(), gate.numel(), self._dt, _lib.stream_ptr(gate.device))
        _lib.check(st, "minf_silu_mul")
        return gate

    def _as_configured(self, hidden):
        """Whether every weight (and the embedded tokens) has the dtype, device and shape that the configuration
        says, the norms' one after the other in memory: what the kernels above take by pointer.  Weights a caller
        filled in otherwise go through torch ops, which promote, broadcast or refuse them; so does a call under
        autocast, whose products come in autocast's dtype."""
        if torch.is_autocast_enabled(self.device.type):
            return False
        c = self.cfg
        qd, kd, inter = c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim, c.intermediate_size
        shapes = {"input_layernorm": (c.hidden_size,), "post_attention_layernorm": (c.hidden_size,),
                  "q_proj": (qd, c.hidden_size), "k_proj": (kd, c.hidden_size), "v_proj": (kd, c.hidden_size),
                  "o_proj": (c.hidden_size, qd), "gate_proj": (inter, c.hidden_size), "up_proj": (inter, c.hidden_size),
                  "down_proj": (c.hidden_size, inter)}

        def fits(t, shape):
            return t.dtype == self.dtype and t.device == hidden.device and tuple(t.shape) == shape \
                and (t.dim() > 1 or t.is_contiguous())
        return self._dt is not None and hidden.is_cuda and fits(hidden, (hidden.shape[0], c.hidden_size)) \
            and fits(self.norm, (c.hidden_size,)) and all(fits(L[k], shape) for L in self.layers for k, shape in shapes.items())

    # ---- prefill --------------------------------------------------------------------------
    @torch.no_grad()
    def prefill(self, input_ids, attn_forward_config=None, chunk=32768, keep_kv=False):
        """input_ids [N] (one sequence).  ``attn_forward_config`` is the reference's dictionary
        (best_pattern per layer/head, starting_layer, minference_ratio); None = every head
        vertical_and_slash (1000, 6096).  Returns (last-token logits [vocab] fp32, kv list or None)."""
        c = self.cfg
        ids = input_ids.to(self.device).reshape(-1)
        n = ids.numel()
        cfg = attn_forward_config if attn_forward_config is not None else {"best_pattern": None}
        hidden = self.embed_tokens[ids]                                    # [N, hidden]
        if not self._as_configured(hidden):
            return self._prefill_torch(hidden, cfg, chunk, keep_kv)
        cos, sin = self._rope_tables(n)
        new = lambda *shape: torch.empty(shape, device=self.device, dtype=self.dtype)
        q, attn = new(n, c.num_heads, c.head_dim), new(n, c.num_heads, c.head_dim)
        # the norm that comes next is taken together with the residual add before it: `normed` holds the
        # input of the next projections
        normed = self._rms(hidden, self.layers[0]["input_layernorm"]) if self.layers else None
        kv_cache = [] if keep_kv else None
        k = v = None
        for li, L in enumerate(self.layers):
            if k is None or keep_kv:
                k, v = new(n, c.num_kv_heads, c.head_dim), new(n, c.num_kv_heads, c.head_dim)
            for s in range(0, n, chunk):
                e = min(s + chunk, n)
                for dst, w in ((q, "q_proj"), (k, "k_proj"), (v, "v_proj")):
                    torch.mm(normed[s:e], L[w].T, out=dst[s:e].view(e - s, -1))
            self._rotate(q, k, cos, sin)
            # [N, H, D] storage viewed as [1, H, N, D]: the kernels take strides, nothing is copied
            minference_prefill_forward(q.permute(1, 0, 2)[None], k.permute(1, 0, 2)[None], v.permute(1, 0, 2)[None],
                                       {"layer_idx": li, "attn_forward_config": cfg, "out": attn.permute(1, 0, 2)[None]})
            nxt = self.layers[li + 1]["input_layernorm"] if li + 1 < len(self.layers) else None
            for s in range(0, n, chunk):
                e = min(s + chunk, n)
                o = attn[s:e].view(e - s, -1) @ L["o_proj"].T
                x = self._rms(hidden[s:e], L["post_attention_layernorm"], delta=o, out=normed[s:e])
                mlp = self._silu_mul(x @ L["gate_proj"].T, x @ L["up_proj"].T) @ L["down_proj"].T
                if nxt is not None:
                    self._rms(hidden[s:e], nxt, delta=mlp, out=normed[s:e])
                else:
                    hidden[s:e] += mlp
            if keep_kv:
                kv_cache.append((k, v))
        last = self._rms(hidden[-1:].clone(), self.norm)
        logits = (last @ self.lm_head.T).float()[0]
        return logits, kv_cache

    def _prefill_torch(self, hidden, cfg, chunk, keep_kv):
        """The same for weights that are not as configured (_as_configured): torch ops around the attention path."""
        c, n = self.cfg, hidden.shape[0]

        def rms(x, weight):
            xf = x.float()
            return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + c.rms_eps)).to(self.dtype) * weight

        def rotate(x, cos, sin):
            half = c.head_dim // 2
            return (x.float() * cos + torch.cat([-x[..., half:], x[..., :half]], dim=-1).float() * sin).to(x.dtype)
        cos, sin = (torch.cat([t, t], dim=-1)[:, None] for t in self._rope_tables(n))
        new = lambda heads: torch.empty((n, heads, c.head_dim), device=self.device, dtype=self.dtype)
        q, k, v, kv_cache = new(c.num_heads), None, None, [] if keep_kv else None
        for li, L in enumerate(self.layers):
            if k is None or keep_kv:
                k, v = new(c.num_kv_heads), new(c.num_kv_heads)
            for s in range(0, n, chunk):
                e = min(s + chunk, n)
                x = rms(hidden[s:e], L["input_layernorm"])
                q[s:e] = rotate((x @ L["q_proj"].T).view(e - s, c.num_heads, c.head_dim), cos[s:e], sin[s:e])
                k[s:e] = rotate((x @ L["k_proj"].T).view(e - s, c.num_kv_heads, c.head_dim), cos[s:e], sin[s:e])
                v[s:e] = (x @ L["v_proj"].T).view(e - s, c.num_kv_heads, c.head_dim)
            attn = minference_prefill_forward(q.permute(1, 0, 2)[None], k.permute(1, 0, 2)[None], v.permute(1, 0, 2)[None],
                                              {"layer_idx": li, "attn_forward_config": cfg})[0].permute(1, 0, 2)
            for s in range(0, n, chunk):
                e = min(s + chunk, n)
                h = hidden[s:e] + attn[s:e].reshape(e - s, -1) @ L["o_proj"].T
                x = rms(h, L["post_attention_layernorm"])
                mlp = (torch.nn.functional.silu(x @ L["gate_proj"].T) * (x @ L["up_proj"].T)) @ L["down_proj"].T
                hidden[s:e] = h + mlp
            if keep_kv:
                kv_cache.append((k, v))
        return (rms(hidden[-1:], self.norm) @ self.lm_head.T).float()[0], kv_cache

    def flops_linear(self, n):
        """FLOPs of the GEMMs of one prefill of n tokens (attention excluded, lm_head on one token)."""
        c = self.cfg
        per_tok = 2 * (c.hidden_size * (c.num_heads + 2 * c.num_kv_heads) * c.head_dim
                       + c.num_heads * c.head_dim * c.hidden_size + 3 * c.hidden_size * c.intermediate_size)
        return c.num_layers * n * per_tok + 2 * c.hidden_size * c.vocab_size


def seeded_pattern_mix(num_layers, num_heads, seed=501, p_vs=0.7, p_bs=0.2,
                       vs=(1000, 6096), ashape=(128, 4096)):
    """BASELINE config 5's per-head pattern table: a seeded mix of vertical_and_slash, block_sparse
    and A-shape heads in the best_pattern format (list over layers of {head: [type, a, b, score]})."""
    import numpy as np
    rng = np.random.default_rng(seed)
    table = []
    for _ in range(num_layers):
        layer = {}
        for h in range(num_heads):
            u = rng.random()
            if u < p_vs:
                layer[str(h)] = ["vertical_and_slash", vs[0], vs[1], 1.0]
            elif u < p_vs + p_bs:
                layer[str(h)] = ["block_sparse", 100, 0, 1.0]
            else:
                layer[str(h)] = ["stream_llm", ashape[0], ashape[1], 1.0]
        table.append(layer)
    return table
