"""Shared building blocks for sharded stage models.

The sharding pattern mirrors the reference (e.g.
/root/reference/shard/server/model/llama.py:26-36): a stage owns a
contiguous [start, end) layer range; the first stage owns embed_tokens,
the last owns the final norm + lm_head.  Unlike the reference we do NOT
materialize IdentityBlock placeholders — layer modules are keyed by
their *global* index in a ModuleDict so weight keys stay globally
consistent without num_hidden_layers dummy entries.
"""

from __future__ import annotations

from typing import Callable, Dict, List, Optional, Tuple

import torch
import torch.nn as nn

from .. import ops
from ..config import ModelConfig, QuantConfig, ShardSpec
from ..ops.kvcache import KVCache

QuantPredicate = Callable[[str], bool]

_READ = set()


def read_in_place(cls):
    """Marks modules whose weights a layer may read in place of a call, or which it may
    call with more than their input."""
    _READ.add(cls)
    return cls


def as_built(*modules) -> bool:
    """Whether these are such modules and nothing depends on their calls: hooks, a
    forward of their own.  (Subclasses are others.)"""
    M = nn.modules.module
    if M._global_forward_hooks or M._global_forward_pre_hooks:
        return False
    for m in modules:
        if type(m) not in _READ:
            return False
        own = m.__dict__
        if own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
            return False
    return not torch.is_grad_enabled() or not (
        M._global_backward_hooks or M._global_backward_pre_hooks
        or any(m._backward_hooks or m._backward_pre_hooks for m in modules))


@read_in_place
class Linear(nn.Module):
    """Dense or MLX-affine-quantized linear, chosen per checkpoint key.

    Dense path → ops.linear: linear_few.hip for up to 64 rows, else
    linear_tiles.hip or the library.  Quantized path → the w4a16/w8a16
    dequant-GEMM op.  Parameter names (weight/scales/biases) match the MLX
    checkpoint layout so pre-quantized checkpoints load directly
    (/root/reference/shard/utils.py:54-65 predicate: a `.scales` key exists
    for the module).
    """

    def __init__(self, in_features: int, out_features: int,
                 quant: Optional[QuantConfig] = None, bias: bool = False,
                 dtype: torch.dtype = torch.bfloat16):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.quant = quant
        if quant is None:
            self.weight = nn.Parameter(
                torch.empty(out_features, in_features, dtype=dtype), requires_grad=False)
        else:
            per_word = 32 // quant.bits
            wdtype = torch.uint32 if hasattr(torch, "uint32") else torch.int32
            self.weight = nn.Parameter(
                torch.empty(out_features, in_features // per_word, dtype=wdtype),
                requires_grad=False)
            self.scales = nn.Parameter(
                torch.empty(out_features, in_features // quant.group_size, dtype=dtype),
                requires_grad=False)
            self.biases = nn.Parameter(
                torch.empty(out_features, in_features // quant.group_size, dtype=dtype),
                requires_grad=False)
        if bias:
            self.bias = nn.Parameter(torch.empty(out_features, dtype=dtype),
                                     requires_grad=False)
        else:
            self.bias = None

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self.quant is None:
            return ops.linear(x, self.weight, self.bias)
        y = ops.quantized_linear(x, self.weight, self.scales, self.biases,
                                 self.quant.group_size, self.quant.bits)
        if self.bias is not None:
            y = y + self.bias
        return y


def dense_weight(m, in_features: int) -> Optional[torch.Tensor]:
    """The weights of a Linear or FusedColumns, packed ones through their bf16 copy;
    None where there is no room for it."""
    q = m.quant
    if q is None:
        return m.weight
    return ops.resident_weight(m.weight, m.scales, m.biases, in_features,
                               q.group_size, q.bits)


def weight_for(m, x: torch.Tensor, in_features: int) -> Optional[torch.Tensor]:
    """dense_weight as ``project`` of rows like x reads it: packed words have a copy only
    on the GPU, and only where torch's own operators are not asked for."""
    return dense_weight(m, in_features) if m.quant is None or ops.use_native(x) else None


def feed(into, out, x: torch.Tensor, act: str, norm: Optional[nn.Module] = None,
         residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The gated unit of ``into``'s halves through ``out``, as ``project`` of each; one
    call for few rows."""
    if into.bias is None and out.bias is None and x.is_cuda:
        w_in = weight_for(into, x, x.shape[-1])
        w_out = weight_for(out, x, sum(into.splits) // 2)
        if w_in is not None and w_out is not None:
            y = ops.feed_few(x, w_in, w_out, act, norm, residual)
            if y is not None:
                return y
    return project(out, project(into, x, norm=norm, act=act), residual=residual)


def attend(qkv, out, x: torch.Tensor, norm: nn.Module, cos, sin, cache, heads: int,
           scale: float, softcap: float = 0.0, window: int = 0,
           residual: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """ops.attend_few with the weights of a FusedColumns and a Linear, or None."""
    w_qkv = weight_for(qkv, x, x.shape[-1])
    w_o = weight_for(out, x, heads * cache.k_head_dim)
    if w_qkv is None or w_o is None:
        return None
    return ops.attend_few(x, w_qkv, qkv.bias, norm, cos, sin, cache, w_o, out.bias, residual,
                          heads, scale, softcap, window)


def project(m, x: torch.Tensor, *, norm: Optional[nn.Module] = None,
            act: Optional[str] = None,
            residual: Optional[torch.Tensor] = None,
            clear: Optional[torch.Tensor] = None) -> torch.Tensor:
    """ops.project with the weights of a Linear or FusedColumns, packed ones
    through their bf16 copy."""
    q, w = m.quant, weight_for(m, x, x.shape[-1])
    if w is not None:
        return ops.project(x, w, m.bias, norm=norm, act=act, residual=residual,
                           clear=clear)
    # no room for the copy, or no kernels
    if clear is not None:
        clear.zero_()
    if norm is not None:
        x = norm(x)
    y = ops.quantized_linear(x, m.weight, m.scales, m.biases, q.group_size,
                             q.bits)
    if m.bias is not None:
        y = y + m.bias
    return ops.finish(y, act, residual)


@read_in_place
class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float = 1e-5, weight_offset: float = 0.0,
                 dtype: torch.dtype = torch.bfloat16):
        super().__init__()
        self.eps = eps
        self.weight_offset = weight_offset
        self.weight = nn.Parameter(torch.ones(dim, dtype=dtype), requires_grad=False)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return ops.rms_norm(x, self.weight, self.eps, self.weight_offset)


read_in_place(nn.Embedding)


def head(norm: nn.Module, x: torch.Tensor, out: Optional[nn.Module] = None,
         table: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out``, or the product with an embedding's rows, of x's normed rows; one kernel
    for few rows.  For 33 to 64 of them and many weights the norm has a kernel of its own
    (2 us of 40 and more; 64 rows, the product alone and the library's: 21720 x 3584 33.8,
    38.6 us; 32000 x 3584 46.0, 44.3; 128256 x 4096 192, 213)."""
    if ops.few_tokens(x) and as_built(norm) and (out is None or as_built(out)):
        V, K = table.shape if out is None else (out.out_features, out.in_features)
        if x.numel() <= 32 * K or V * K <= 1 << 26:
            if out is None:
                return ops.project(x, table, norm=norm)
            return project(out, x, norm=norm)
    x = norm(x)
    return ops.linear(x, table) if out is None else out(x)


class StageModel(nn.Module):
    """Base class for one pipeline stage of a sharded model.

    Subclasses set up, inside ``self.model`` (an inner module named so
    state-dict keys match the checkpoint's ``model.*`` prefix):
      - ``embed_tokens`` when the shard owns it
      - ``layers``: ModuleDict {str(global_idx): DecoderLayer}
      - ``norm`` when last
    and ``self.lm_head`` when last (or tie to embeddings).
    """

    rope_attn_scale: float = 1.0
    # runs ragged batches over a PagedState (``run``, ``make_state``)
    supports_ragged: bool = False
    supports_quantization: bool = True

    def __init__(self, config: ModelConfig, shard: ShardSpec):
        super().__init__()
        self.config = config
        self.shard = shard
        self._rt_len = 0
        self._rt_dev = None
        self._rt_old: List[Tuple[torch.Tensor, torch.Tensor]] = []

    # -- RoPE tables -------------------------------------------------------
    def _rope_tables(self, device, min_len: int):
        """Host-precomputed cos/sin tables [N, D/2] fp32 (guide Appendix B:
        no per-element trig on device); grown lazily, device-resident."""
        if self._rt_len < min_len or self._rt_dev != device:
            n = max(1024, 1 << max(int(min_len) - 1, 1).bit_length())
            if self._rt_len:  # captured graphs may still read the old ones
                self._rt_old.append((self._rt_cos, self._rt_sin))
            pos = torch.arange(n, device=device)
            inv = self.rope_inv_freq.to(device)
            from .. import ops as _ops
            cos, sin = _ops.rope_cos_sin(pos, inv, self.rope_attn_scale)
            self._rt_cos = cos.contiguous()
            self._rt_sin = sin.contiguous()
            self._rt_len, self._rt_dev = n, device
        return self._rt_cos, self._rt_sin

    def begin(self, x: torch.Tensor, cache, embed: Optional[nn.Module] = None,
              scale: Optional[torch.Tensor] = None):
        """(hidden states, cos, sin) of this forward: x, or its rows of ``embed``
        (times ``scale``), and its positions' rotations."""
        first = cache[0] if cache else None
        if embed is None:
            h = x
        else:
            pos = first.graph_pos if first is not None else None
            if (pos is not None and x.shape[1] == 1 and type(embed) is nn.Embedding
                    and as_built(embed) and embed.max_norm is None
                    and getattr(self.rope_for, "__func__", None) is StageModel.rope_for):
                found = ops.step_begin(x, embed.weight, scale, pos,
                                       *self._rope_tables(x.device, first.capacity))
                if found is not None:
                    return found
            h = embed(x)
            if scale is not None:
                h = h * scale.to(h.dtype)
        cos, sin, _ = self.rope_for(first, h.shape[1], h.device)
        return h, cos, sin

    def rope_for(self, cache0, T: int, device):
        """(cos, sin, offset) for this forward; handles graph-pos mode
        (device position tensor) and the eager python-offset mode."""
        gp = cache0.graph_pos if cache0 is not None else None
        if gp is not None:
            cos_t, sin_t = self._rope_tables(device, cache0.capacity)
            idx = gp.to(torch.long)
            return cos_t.index_select(0, idx), sin_t.index_select(0, idx), 0
        offset = cache0.offset if cache0 is not None else 0
        cos_t, sin_t = self._rope_tables(device, offset + T)
        return cos_t[offset: offset + T], sin_t[offset: offset + T], offset

    @property
    def fp_dtype(self) -> torch.dtype:
        """Activation dtype = first floating parameter's dtype (a packed
        uint32 quant weight can come first on stages without embeddings
        — casting activations to THAT truncates them to garbage)."""
        return next((q.dtype for q in self.parameters()
                     if q.is_floating_point()), torch.bfloat16)

    @property
    def hop_dtype(self) -> torch.dtype:
        """Type of the hidden states handed from stage to stage."""
        return self.fp_dtype

    @property
    def hop_width(self) -> int:
        """Width of what this stage takes from the previous one."""
        return self.config.hidden_size

    @classmethod
    def allowed_cuts(cls, config: ModelConfig) -> Optional[List[int]]:
        """Layer indices a stage may begin at; None: any."""
        return None

    # -- cache ------------------------------------------------------------
    def cache_specs(self) -> List[Tuple[int, int, int]]:
        """(n_kv_heads, k_head_dim, v_head_dim) for each *owned* layer."""
        raise NotImplementedError

    def make_cache(self, dtype: Optional[torch.dtype] = None, batch_size: int = 1,
                   device=None) -> List[KVCache]:
        # dtype from the first FLOATING parameter: on a quantized stage
        # without embeddings the first parameter is a packed uint32
        # weight, and a uint32 KV cache silently truncates every K/V
        # value to zero (caught as PP-parity divergence)
        every = self.parameters()
        p = next(every)
        fp = p if p.is_floating_point() else next(
            (q for q in every if q.is_floating_point()), p)
        from ..ops.kvcache import make_cache
        return make_cache(self.cache_specs(),
                          dtype=dtype or fp.dtype,
                          device=device if device is not None else p.device,
                          batch_size=batch_size)

    # -- weights ----------------------------------------------------------
    @classmethod
    def complete_config(cls, config: ModelConfig,
                        weights: Dict[str, torch.Tensor]):
        """Enter sizes that only the checkpoint's tensors tell."""

    @classmethod
    def owns_key(cls, key: str, shard: ShardSpec) -> bool:
        """Key-routing rule — identical to the reference splitter
        (/root/reference/sharding_weight.py:17-24): layer keys by index
        range, embeddings on the first shard, final norm + lm_head on
        the last."""
        if key.startswith("model.layers."):
            idx = int(key.split(".")[2])
            return shard.owns(idx)
        if key.startswith("model.embed_tokens"):
            return shard.is_first
        if key.startswith("model.norm") or key.startswith("lm_head"):
            return shard.is_last
        return False

    @classmethod
    def sanitize(cls, weights: Dict[str, torch.Tensor], shard: ShardSpec) -> Dict[str, torch.Tensor]:
        """Filter a merged weight dict down to this shard's keys and drop
        buffers that are recomputed (rotary inv_freq), matching
        /root/reference/shard/server/model/llama.py:92-107."""
        return {k: v for k, v in weights.items()
                if cls.owns_key(k, shard) and "rotary_emb.inv_freq" not in k}

    def load_weights(self, weights: Dict[str, torch.Tensor], strict: bool = True):
        weights = self.sanitize(weights, self.shard)
        missing, unexpected = self.load_state_dict(weights, strict=False)
        # tied lm_head shows up as missing when the checkpoint ties embeddings
        missing = [m for m in missing if not self._key_optional(m)]
        if strict and (missing or unexpected):
            raise RuntimeError(
                f"weight mismatch: missing={missing[:8]} unexpected={unexpected[:8]}")
        return missing, unexpected

    def _key_optional(self, key: str) -> bool:
        return False

    # -- forward ----------------------------------------------------------
    def forward(self, x: torch.Tensor, cache: Optional[List[KVCache]] = None) -> torch.Tensor:
        """x: [B, T] int64 token ids on the first shard, else [B, T, H]
        hidden states.  Returns hidden states, or logits on the last shard."""
        raise NotImplementedError


def owned_layer_indices(shard: ShardSpec) -> List[int]:
    return list(range(shard.start_layer, shard.end_layer))
