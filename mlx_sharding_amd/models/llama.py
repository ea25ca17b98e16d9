"""Llama-family stage model (covers Mistral via the model_type remap).

Capability parity with /root/reference/shard/server/model/llama.py:
same shard semantics (embed on first, norm+lm_head on last, tied
embeddings via lm_head fallback), same key routing; compute runs on
our op layer (HIP kernels on GPU, torch reference on CPU).
"""

from __future__ import annotations

from typing import List, Optional, Tuple

import torch
import torch.nn as nn

from .. import ops
from ..config import ModelConfig, ShardSpec
from ..ops.kvcache import KVCache
from .base import (Linear, RMSNorm, StageModel, as_built, attend, feed, head,
                   owned_layer_indices, project, read_in_place, weight_for)


@read_in_place
class LlamaAttention(nn.Module):
    def __init__(self, cfg: ModelConfig, quant_for, prefix: str):
        super().__init__()
        H = cfg.hidden_size
        self.n_heads = cfg["num_attention_heads"]
        self.n_kv_heads = cfg.get("num_key_value_heads", self.n_heads)
        self.head_dim = cfg.get("head_dim") or H // self.n_heads
        self.scale = self.head_dim ** -0.5
        # qwen2 (served through this class via MODEL_REMAPPING) hardcodes
        # QKV bias on / o_proj bias off in its HF reference; llama-family
        # configs carry an explicit attention_bias flag for all four
        qkv_bias = bool(cfg.get("attention_bias", cfg.model_type == "qwen2"))
        o_bias = bool(cfg.get("attention_bias", False))
        q = lambda name: quant_for(f"{prefix}.{name}")
        self.q_proj = Linear(H, self.n_heads * self.head_dim, q("q_proj"), qkv_bias)
        self.k_proj = Linear(H, self.n_kv_heads * self.head_dim, q("k_proj"), qkv_bias)
        self.v_proj = Linear(H, self.n_kv_heads * self.head_dim, q("v_proj"), qkv_bias)
        self.o_proj = Linear(self.n_heads * self.head_dim, H, q("o_proj"), o_bias)
        self._fused_qkv = None  # set by fuse_model()

    def read(self):
        """Modules that are read in place of a call where few tokens come."""
        m = self._modules
        if self._fused_qkv is not None:
            return (m["o_proj"],)
        return m["q_proj"], m["k_proj"], m["v_proj"], m["o_proj"]

    def forward(self, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                cache: Optional[KVCache], norm: Optional[RMSNorm] = None,
                residual: Optional[torch.Tensor] = None) -> torch.Tensor:
        """norm: for x's rows first; residual: added to what is returned.  For
        few tokens, where both go with the projections."""
        B, T, _ = x.shape
        if (T > 1 and norm is not None and self._fused_qkv is not None
                and type(cache) is KVCache and as_built(self.o_proj)):
            out = attend(self._fused_qkv, self.o_proj, x, norm, cos, sin, cache, self.n_heads,
                         self.scale, residual=residual)
            if out is not None:
                return out
        if self._fused_qkv is not None and norm is not None:
            q, k, v = project(self._fused_qkv, x, norm=norm).split(
                self._fused_qkv.splits, -1)
        elif self._fused_qkv is not None:
            q, k, v = self._fused_qkv(x)
        elif norm is not None:
            q, k, v = (project(m, x, norm=norm)
                       for m in (self.q_proj, self.k_proj, self.v_proj))
        else:
            q, k, v = self.q_proj(x), self.k_proj(x), self.v_proj(x)
        q = q.view(B, T, self.n_heads, self.head_dim)
        k = k.view(B, T, self.n_kv_heads, self.head_dim)
        v = v.view(B, T, self.n_kv_heads, self.head_dim)
        offset = 0
        gp = None
        out = None
        if T == 1 and type(cache) is KVCache:  # others append by methods of their own
            ahead = None  # a hint, for the few sequences that it is for
            if B <= 16 and as_built(self.o_proj):
                ahead = weight_for(self.o_proj, x, self.n_heads * self.head_dim)
            out = cache.attend_step(q, k, v, cos, sin, self.scale, faster=True, ahead=ahead)
        if out is not None:
            pass
        elif cache is not None and ops.use_native(x):
            # both rotations and the scatter into the caches in one kernel
            gp = cache.graph_pos
            if gp is None:
                offset = cache.offset
            q, k, v = cache.append_rope_qkv(q, k, v, cos, sin)
        else:
            q = ops.apply_rope(q, cos, sin)
            k = ops.apply_rope(k, cos, sin).transpose(1, 2)
            v = v.transpose(1, 2)
            if cache is not None:
                gp = cache.graph_pos
                if gp is None:
                    offset = cache.offset
                k, v = cache.update(k, v)
        if out is None:
            out = ops.attention(q.transpose(1, 2), k, v, self.scale,
                                causal_offset=offset, pos_dev=gp)
            out = out.transpose(1, 2).reshape(B, T, -1)
        if residual is not None:
            return project(self.o_proj, out, residual=residual)
        return self.o_proj(out)


@read_in_place
class LlamaMLP(nn.Module):
    def __init__(self, cfg: ModelConfig, quant_for, prefix: str):
        super().__init__()
        H = cfg.hidden_size
        I = cfg["intermediate_size"]
        q = lambda name: quant_for(f"{prefix}.{name}")
        self.gate_proj = Linear(H, I, q("gate_proj"))
        self.up_proj = Linear(H, I, q("up_proj"))
        self.down_proj = Linear(I, H, q("down_proj"))
        self._fused_gu = None  # set by fuse_model()

    def read(self):
        """As in LlamaAttention."""
        return (self._modules["down_proj"],)

    def forward(self, x: torch.Tensor, norm: Optional[RMSNorm] = None,
                residual: Optional[torch.Tensor] = None) -> torch.Tensor:
        """norm, residual: as in LlamaAttention."""
        if self._fused_gu is not None and (
                norm is not None or (ops.few_tokens(x) and as_built(self.down_proj))):
            return feed(self._fused_gu, self.down_proj, x, "silu", norm, residual)
        if norm is not None:
            x = norm(x)
        if residual is not None:
            return residual + self(x)
        if self._fused_gu is not None:
            return self.down_proj(project(self._fused_gu, x, act="silu"))
        return self.down_proj(ops.swiglu(self.gate_proj(x), self.up_proj(x)))


class LlamaDecoderLayer(nn.Module):
    def __init__(self, cfg: ModelConfig, quant_for, prefix: str):
        super().__init__()
        eps = cfg.get("rms_norm_eps", 1e-5)
        self.self_attn = LlamaAttention(cfg, quant_for, f"{prefix}.self_attn")
        self.mlp = LlamaMLP(cfg, quant_for, f"{prefix}.mlp")
        self.input_layernorm = RMSNorm(cfg.hidden_size, eps)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, eps)

    def forward(self, x, cos, sin, cache):
        attn, mlp, norm = self.self_attn, self.mlp, self.input_layernorm
        if (ops.few_tokens(x) and as_built(attn, mlp, norm)
                and as_built(*attn.read(), *mlp.read())):
            h = attn(x, cos, sin, cache, norm, x)
            return mlp(h, self.post_attention_layernorm, h)
        pn, H = self.post_attention_layernorm, x.shape[-1]
        more = ops.more_tokens(x)  # of which each half of the layer may be as few
        if (more and x.shape[1] > 1 and type(cache) is KVCache and as_built(attn, norm)
                and as_built(*attn.read()) and attn._fused_qkv is not None
                and ops.one_round(x, (sum(attn._fused_qkv.splits), H, None),
                                  (H, attn.n_heads * attn.head_dim, None))):
            h, y = attn(x, cos, sin, cache, norm, x), None
        else:
            # fused: h = x + attn; y = rms_norm(h) in one kernel
            y, h = ops.rms_norm_residual(attn(norm(x), cos, sin, cache), x, pn.weight,
                                         pn.eps, pn.weight_offset)
        if (y is None and as_built(mlp, pn) and as_built(*mlp.read())
                and mlp._fused_gu is not None
                and ops.one_round(h, (sum(mlp._fused_gu.splits) // 2, H, "silu"),
                                  (H, sum(mlp._fused_gu.splits) // 2, None))):
            return mlp(h, pn, h)
        if y is None:
            y = pn(h)
        return h + mlp(y)


class _Inner(nn.Module):
    pass


class LlamaStageModel(StageModel):
    model_type = "llama"

    def __init__(self, config: ModelConfig, shard: ShardSpec, quant_for=None):
        super().__init__(config, shard)
        quant_for = quant_for or (lambda prefix: None)
        H = config.hidden_size
        self.model = _Inner()
        if shard.is_first:
            self.model.embed_tokens = nn.Embedding(config.vocab_size, H,
                                                   dtype=torch.bfloat16)
        layers = nn.ModuleDict()
        for i in owned_layer_indices(shard):
            layers[str(i)] = LlamaDecoderLayer(config, quant_for, f"model.layers.{i}")
        self.model.layers = layers
        self.tie_word_embeddings = bool(config.get("tie_word_embeddings", False))
        if shard.is_last:
            self.model.norm = RMSNorm(H, config.get("rms_norm_eps", 1e-5))
            if not self.tie_word_embeddings:
                self.lm_head = Linear(H, config.vocab_size, quant_for("lm_head"))
            elif not shard.is_first:
                # tied head needs the embedding table on the last shard too
                self.model.embed_tokens = nn.Embedding(config.vocab_size, H,
                                                       dtype=torch.bfloat16)
        head_dim = config.get("head_dim") or H // config["num_attention_heads"]
        inv = ops.rope_freqs(head_dim, float(config.get("rope_theta", 10000.0)),
                             config.get("rope_scaling"))
        self.register_buffer("rope_inv_freq", inv, persistent=False)

    def _key_optional(self, key: str) -> bool:
        # a tied checkpoint may or may not carry lm_head.weight
        return key.startswith("lm_head") and self.tie_word_embeddings

    def cache_specs(self) -> List[Tuple[int, int, int]]:
        cfg = self.config
        hd = cfg.get("head_dim") or cfg.hidden_size // cfg["num_attention_heads"]
        nkv = cfg.get("num_key_value_heads", cfg["num_attention_heads"])
        return [(nkv, hd, hd) for _ in range(self.shard.n_layers)]

    def forward(self, x: torch.Tensor, cache: Optional[List[KVCache]] = None) -> torch.Tensor:
        h, cos, sin = self.begin(
            x, cache, self.model.embed_tokens if self.shard.is_first else None)
        for j, i in enumerate(owned_layer_indices(self.shard)):
            c = cache[j] if cache is not None else None
            h = self.model.layers[str(i)](h, cos, sin, c)
        if self.shard.is_last:
            if self.tie_word_embeddings:
                h = head(self.model.norm, h, table=self.model.embed_tokens.weight)
            else:
                h = head(self.model.norm, h, self.lm_head)
        return h
