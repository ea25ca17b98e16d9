"""A layer's attention of few tokens in one call, beside the same kernels one by one."""

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.models.base import RMSNorm
from mlx_sharding_amd.ops.kvcache import KVCache

pytestmark = pytest.mark.gpu


def one_by_one(x, w, b, norm, cos, sin, cache, wo, bo, res, heads, scale, cap, window):
    B, T, _ = x.shape
    D = cache.k_head_dim
    at = cache.offset
    y = ops.project(x, w, b, norm=norm)
    q, k, v = (t.view(B, T, -1, D) for t in y.split(
        [heads * D, cache.n_kv_heads * D, cache.n_kv_heads * D], -1))
    q, k, v = cache.append_rope_qkv(q, k, v, cos, sin)
    o = ops.attention(q.transpose(1, 2), k, v, scale, causal_offset=at, softcap=cap,
                      sliding_window=window)
    return ops.project(o.transpose(1, 2).reshape(B, T, -1), wo, bo, residual=res)


def inputs(B, T, H, heads, kv, D, bias, dtype=torch.bfloat16):
    g = torch.Generator("cuda").manual_seed(T + heads)

    def new(*n):
        return torch.randn(*n, generator=g, device="cuda").to(dtype)

    wide = (heads + 2 * kv) * D
    norm = RMSNorm(H, 1e-5, 1.0).cuda()
    norm.weight.data = new(H) * 0.1
    angle = torch.rand(T, D // 2, generator=g, device="cuda")
    return dict(x=new(B, T, H), w=new(wide, H) * H ** -0.5, b=new(wide) if bias else None,
                norm=norm, cos=torch.cos(angle), sin=torch.sin(angle),
                wo=new(H, heads * D) * H ** -0.5, bo=new(H) if bias else None,
                res=new(B, T, H) if bias else None)


def cache_of(B, kv, D, at, dtype=torch.bfloat16):
    cache = KVCache(kv, D, D, device="cuda", batch_size=B, dtype=dtype)
    if at:
        g = torch.Generator("cuda").manual_seed(at)
        cache.update(*(torch.randn(B, kv, at, D, generator=g, device="cuda").to(dtype)
                       for _ in range(2)))
    return cache


@torch.no_grad()
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("B,T,H,heads,kv,D,at,cap,window", [
    (1, 2, 64, 2, 1, 32, 0, 0.0, 0), (1, 64, 256, 4, 4, 64, 0, 0.0, 0),
    (1, 57, 256, 8, 2, 64, 1000, 0.0, 0), (5, 11, 128, 4, 2, 128, 9, 0.0, 0),
    (1, 33, 512, 4, 2, 256, 70, 50.0, 40), (32, 2, 96, 3, 1, 64, 3, 0.0, 0)])
def test_same_as_one_by_one(B, T, H, heads, kv, D, at, cap, window, bias):
    a = inputs(B, T, H, heads, kv, D, bias)
    args = (heads, D ** -0.5, cap, window)
    here, there = cache_of(B, kv, D, at), cache_of(B, kv, D, at)
    got = ops.attend_few(a["x"], a["w"], a["b"], a["norm"], a["cos"], a["sin"], here,
                         a["wo"], a["bo"], a["res"], *args)
    want = one_by_one(a["x"], a["w"], a["b"], a["norm"], a["cos"], a["sin"], there, a["wo"],
                      a["bo"], a["res"], *args)
    assert got.shape == a["x"].shape and torch.equal(got, want)
    assert here.offset == there.offset == at + T
    assert torch.equal(here.k, there.k) and torch.equal(here.v, there.v)


@torch.no_grad()
def test_what_is_left_to_the_others():
    a = inputs(1, 9, 128, 4, 2, 64, True)

    def call(cache=None, **other):
        b = {**a, **other}
        cache = cache or cache_of(1, 2, 64, 5)
        was = cache.offset
        out = ops.attend_few(b["x"], b["w"], b["b"], b["norm"], b["cos"], b["sin"], cache,
                             b["wo"], b["bo"], b["res"], 4, 0.125, 0.0, 0)
        assert cache.offset == (was if out is None else was + b["x"].shape[1])
        return out

    assert call() is not None
    many = inputs(1, 65, 128, 4, 2, 64, True)
    assert call(**many) is None
    assert call(cache_of(1, 2, 64, 5, torch.float32)) is None
    assert call(x=a["x"].float()) is None
    assert call(b=a["b"][:-1]) is None
    assert call(w=a["w"][:-64], b=None) is None
    assert call(cos=a["cos"].double()) is None
    assert call(cos=a["cos"][:, :16], sin=a["sin"][:, :16]) is None
    assert call(res=a["res"][:, :1]) is None
    assert call(res=a["res"].expand(2, -1, -1)) is None
    captured = cache_of(1, 2, 64, 5)
    captured.graph_pos = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert call(captured) is None
    with torch.enable_grad():
        assert call(x=a["x"].clone().requires_grad_()) is None
