"""Per-layer KV cache: preallocated contiguous, grow-by-chunk.

Layout [B, n_kv_heads, S, D] with independent K and V head dims (MLA
stores K at qk_nope+qk_rope=192 and V at 128 — the tuple head_dim the
reference exposes at /root/reference/shard/server/model/deepseek_v2.py:120-125).

The reference's cache lifecycle: one fresh cache per
generation request, exactly one multi-token prefill then T=1 decode
steps.  Sessions own their caches here (no global mutable CACHE).
"""

from __future__ import annotations

from typing import List, Optional, Tuple

import torch


class KVCache:
    CHUNK = 1024

    def __init__(self, n_kv_heads: int, k_head_dim: int, v_head_dim: int,
                 dtype: torch.dtype = torch.bfloat16,
                 device: torch.device | str = "cpu",
                 batch_size: int = 1):
        self.n_kv_heads = n_kv_heads
        self.k_head_dim = k_head_dim
        self.v_head_dim = v_head_dim
        # an integer cache dtype silently truncates K/V on copy (torch
        # casts without complaint) — fail loudly instead
        if not dtype.is_floating_point:
            raise TypeError(f"KV cache dtype must be floating, got {dtype}")
        self.dtype = dtype
        self.device = torch.device(device)
        self.batch_size = batch_size
        self.offset = 0
        self._k: Optional[torch.Tensor] = None
        self._v: Optional[torch.Tensor] = None
        # zeros that attend_step's kernel counts its blocks with, and leaves as zeros;
        # made for tokens, as a prompt has no need of them
        self._tickets: Optional[torch.Tensor] = None
        # hipGraph-captured decode: position lives on device (int32 [1]);
        # update() appends by index_copy_ and python offset is not advanced.
        self.graph_pos: Optional[torch.Tensor] = None

    def _ensure(self, batch: int, needed: int):
        cap = 0 if self._k is None else self._k.shape[2]
        if self._k is not None and self._k.shape[0] != batch:
            raise ValueError(f"KV cache batch mismatch: {self._k.shape[0]} vs {batch}")
        if needed <= cap and self._k is not None:
            return
        new_cap = ((needed + self.CHUNK - 1) // self.CHUNK) * self.CHUNK
        nk = torch.empty(batch, self.n_kv_heads, new_cap, self.k_head_dim,
                         dtype=self.dtype, device=self.device)
        nv = torch.empty(batch, self.n_kv_heads, new_cap, self.v_head_dim,
                         dtype=self.dtype, device=self.device)
        if self._k is not None and self.offset > 0:
            nk[:, :, : self.offset] = self._k[:, :, : self.offset]
            nv[:, :, : self.offset] = self._v[:, :, : self.offset]
        self._k, self._v = nk, nv

    def update(self, k: torch.Tensor, v: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
        """Append k/v [B, n_kv, T, D]; return full views [B, n_kv, offset+T, D].

        In graph mode (graph_pos set) the append is an index_copy_ at the
        device position and the FULL buffers are returned — the caller
        passes graph_pos to the attention op, which reads the length on
        device (capture-safe: no python-int shapes)."""
        if self.graph_pos is not None:
            idx = self.graph_pos.to(torch.long)
            self._k.index_copy_(2, idx, k)
            self._v.index_copy_(2, idx, v)
            return self._k, self._v
        B, H, T, _ = k.shape
        self._ensure(B, self.offset + T)
        self._k[:, :, self.offset: self.offset + T] = k
        self._v[:, :, self.offset: self.offset + T] = v
        self.offset += T
        return (self._k[:, :, : self.offset], self._v[:, :, : self.offset])

    def append_mla(self, kvh: torch.Tensor, kpe: torch.Tensor):
        """Fused MLA append: kvh [B, T, nh, nope+vd] (kv_b output) and
        roped kpe [B, T, rope] scatter straight into the caches — no
        cat/head-expand/index_copy round trips.  GPU-only (the HIP
        extension provides the kernel); returns (k, v) like update()."""
        from .. import ops as _ops
        ext = _ops.hip_ext()
        B, T = kvh.shape[0], kvh.shape[1]
        if self.graph_pos is not None:
            ext.mla_append_kv(kvh, kpe, self._k, self._v,
                              pos=self.graph_pos)
            return self._k, self._v
        self._ensure(B, self.offset + T)
        ext.mla_append_kv(kvh, kpe, self._k, self._v, pos0=self.offset)
        self.offset += T
        return (self._k[:, :, : self.offset], self._v[:, :, : self.offset])

    def claim(self, batch: int, T: int):
        """Places for T more rows, for a kernel that writes them itself:
        (position on the device or None, first place).  The rows count from
        ``wrote`` on, when the kernel has been launched."""
        if self.graph_pos is not None:
            return self.graph_pos, 0
        self._ensure(batch, self.offset + T)
        return None, self.offset

    def wrote(self, T: int):
        if self.graph_pos is None:
            self.offset += T

    def attend_step(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                    cos: torch.Tensor, sin: torch.Tensor, scale: float,
                    softcap: float = 0.0, window: int = 0, faster: bool = False,
                    ahead: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
        """append_rope_qkv of one token per sequence and its attention in one kernel:
        [B, 1, heads * D]; None (and nothing appended) where that does not take it, or,
        asked for what is ``faster``, where the separate kernels are.  ahead: weights of
        the product behind it, which are fetched meanwhile."""
        from .. import ops as _ops
        if not (self.dtype == torch.bfloat16 and k.shape[1] == 1
                and self.k_head_dim == self.v_head_dim == k.shape[3]
                and _ops.use_native(q) and all(_ops.plain(t) for t in (q, k, v))):
            return None
        pos, at = self.claim(k.shape[0], 1)
        if self._tickets is None:
            if torch.cuda.is_current_stream_capturing():
                return None  # the zeros would be written by replays only
            self._make_tickets()
        out = _ops.hip_ext().attn_step(q, k, v, cos, sin, self._k, self._v, pos, at,
                                       self._tickets, scale, softcap, window, faster,
                                       ahead)
        if out is not None:
            self.wrote(1)
        return out

    def append_rope_kv(self, k: torch.Tensor, v: torch.Tensor,
                       cos: torch.Tensor, sin: torch.Tensor,
                       interleaved: bool = False):
        """Fused GQA append: RoPE the new k rows [B, T, Hkv, D] and
        scatter k/v straight into the caches (replaces a rope launch +
        two index_copy launches).  GPU-only; returns (k, v) like
        update()."""
        from .. import ops as _ops
        ext = _ops.hip_ext()
        B, T = k.shape[0], k.shape[1]
        if self.graph_pos is not None:
            ext.rope_append_kv(k, v, cos, sin, self._k, self._v,
                               pos=self.graph_pos, interleaved=interleaved)
            return self._k, self._v
        self._ensure(B, self.offset + T)
        ext.rope_append_kv(k, v, cos, sin, self._k, self._v,
                           pos0=self.offset, interleaved=interleaved)
        self.offset += T
        return (self._k[:, :, : self.offset], self._v[:, :, : self.offset])

    def append_rope_qkv(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                        cos: torch.Tensor, sin: torch.Tensor):
        """append_rope_kv with the queries turned as well: (q, k, v).  One kernel where
        heads of a row lie side by side in whole 16-byte vectors."""
        from .. import ops as _ops
        B, T, _, D = k.shape
        if not (D % 16 == 0 and self.k_head_dim == self.v_head_dim == D
                and self.dtype == torch.bfloat16 and cos.dtype == torch.float32
                and all(t.dtype == torch.bfloat16 and t.stride(3) == 1
                        and t.stride(2) == D and t.data_ptr() % 16 == 0
                        # one token each: the stride between tokens says nothing
                        and (t.stride(0) % 8 == 0 if T == 1 else
                             t.stride(1) % 8 == 0
                             and (B == 1 or t.stride(0) == T * t.stride(1)))
                        for t in (q, k, v))):
            q = _ops.apply_rope(q, cos, sin)
            return (q, *self.append_rope_kv(k, v, cos, sin))
        pos, at = self.claim(B, T)
        q = _ops.hip_ext().rope_qkv(q, k, v, cos.contiguous(), sin.contiguous(),
                                    self._k, self._v, pos, at)
        self.wrote(T)
        if pos is not None:
            return q, self._k, self._v
        return q, self._k[:, :, : self.offset], self._v[:, :, : self.offset]

    @property
    def k(self) -> Optional[torch.Tensor]:
        return None if self._k is None else self._k[:, :, : self.offset]

    @property
    def v(self) -> Optional[torch.Tensor]:
        return None if self._v is None else self._v[:, :, : self.offset]

    def keys_buffer(self) -> Optional[torch.Tensor]:
        """Full backing buffer (for the HIP decode kernel, which indexes by offset)."""
        return self._k

    def values_buffer(self) -> Optional[torch.Tensor]:
        return self._v

    @property
    def capacity(self) -> int:
        return 0 if self._k is None else self._k.shape[2]

    def ensure_capacity(self, cap: int, batch: Optional[int] = None):
        b = batch if batch is not None else (
            self._k.shape[0] if self._k is not None else self.batch_size)
        self._ensure(b, cap)
        # a capture's warm-up steps run on a stream of their own
        self._make_tickets()

    def _make_tickets(self):
        if self._tickets is None and self._k is not None and self._k.is_cuda:
            self._tickets = torch.zeros(self._k.shape[0] * self.n_kv_heads,
                                        dtype=torch.int32, device=self._k.device)

    # a shorter prefix of what is cached can be returned to
    trimmable = True

    def snapshot(self):
        """What a decode step changes besides appending; nothing here."""
        return None

    def restore(self, snap):
        pass

    def trim(self, n: int):
        """Roll back to the first ``n`` cached positions (prefix-cache
        reuse: a follow-up request whose prompt shares an n-token prefix
        with the previous generation re-uses those K/V rows and only
        prefills the tail)."""
        if n < 0 or n > self.offset:
            raise ValueError(f"trim({n}) outside [0, {self.offset}]")
        self.offset = n
        self.graph_pos = None

    def reset(self):
        self.offset = 0
        self.graph_pos = None


def make_cache(layer_specs: List[Tuple[int, int, int]], dtype: torch.dtype,
               device, batch_size: int = 1) -> List[KVCache]:
    """Build one KVCache per (n_kv_heads, k_dim, v_dim) layer spec."""
    return [KVCache(h, kd, vd, dtype=dtype, device=device, batch_size=batch_size)
            for (h, kd, vd) in layer_specs]
