"""A token's rotations, cache rows and attention in one kernel, beside the separate ones
and against 64 bits."""

import math

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.ops.kvcache import KVCache

pytestmark = pytest.mark.gpu


def _caches(B, Hkv, D, cached, room, captured, gen):
    made = []
    for _ in range(2):
        c = KVCache(Hkv, D, D, torch.bfloat16, torch.device("cuda"))
        c._ensure(B, room)
        c._k.fill_(math.nan)
        c._v.fill_(math.nan)
        made.append(c)
    one, two = made
    for t in ("_k", "_v"):
        rows = torch.randn(B, Hkv, cached, D, generator=gen, device="cuda").bfloat16()
        for c in made:
            getattr(c, t)[:, :, :cached] = rows
    for c in made:
        c.offset = cached
        if captured:
            c.graph_pos = torch.tensor([cached], dtype=torch.int32, device="cuda")
    return made


def _token(B, Hq, Hkv, D, gen):
    rows = torch.randn(B, 1, (Hq + 2 * Hkv) * D, generator=gen, device="cuda").bfloat16()
    angle = torch.rand(1, D // 2, generator=gen, device="cuda") * 2 * math.pi
    return ([t.view(B, 1, -1, D) for t in rows.split([Hq * D, Hkv * D, Hkv * D], -1)],
            torch.cos(angle), torch.sin(angle))


def _exact(q, cos, sin, keys, values, cap, window):
    """Attention in 64 bits of a query, turned and rounded, to keys [B, Hkv, S, D]."""
    B, _, Hq, D = q.shape
    a, b = q.double().chunk(2, -1)
    c, s = cos.double(), sin.double()
    q = torch.cat([a * c - b * s, b * c + a * s], -1).bfloat16().double()
    if window:
        keys, values = keys[:, :, -window:], values[:, :, -window:]
    k, v = (t.double().repeat_interleave(Hq // t.shape[1], 1) for t in (keys, values))
    z = (k @ q.transpose(1, 2).transpose(2, 3)).squeeze(-1) * 0.1
    if cap:
        z = cap * torch.tanh(z / cap)
    return (torch.softmax(z, -1)[:, :, None] @ v).reshape(B, 1, -1)


# no key before, the token first, last and in the middle of a tile, one slice and 64,
# slices without keys (captured ones are made for the whole room)
@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("window,cap", [(0, 0.0), (70, 30.0)])
@pytest.mark.parametrize("B,Hq,Hkv,D,cached", [
    (1, 1, 1, 64, 0), (1, 32, 4, 64, 63), (1, 32, 8, 128, 64), (3, 14, 2, 128, 1023),
    (64, 32, 8, 128, 100), (5, 16, 8, 256, 31), (1, 16, 1, 256, 2000), (2, 2, 2, 256, 32),
    (1, 2, 1, 128, 5000)])
def test_same_as_separate_kernels(B, Hq, Hkv, D, cached, window, cap, captured):
    g = torch.Generator("cuda").manual_seed(cached + D)
    one, two = _caches(B, Hkv, D, cached, cached + 40, captured, g)
    for step in range(3):
        (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
        got = one.attend_step(q, k, v, cos, sin, 0.1, cap, window)
        gp, at = two.graph_pos, two.offset
        qt, kt, vt = two.append_rope_qkv(q, k, v, cos, sin)
        want = ops.attention(qt.transpose(1, 2), kt, vt, 0.1, causal_offset=at,
                             softcap=cap, sliding_window=window, pos_dev=gp)
        assert one.offset == two.offset
        # a turn's two products may be contracted the other way round: one bf16 step in
        # a key or query
        for a, b in ((one._k, two._k), (one._v, two._v)):
            assert torch.allclose(a.float(), b.float(), rtol=2.0 ** -7, atol=1e-6,
                                  equal_nan=True)
        want = want.transpose(1, 2).reshape(B, 1, -1)
        assert got.shape == want.shape
        assert float((got.float() - want.float()).norm() / want.float().norm()) < 2e-3
        exact = _exact(q, cos, sin, *(t[:, :, : cached + step + 1] for t in (one._k, one._v)),
                       cap, window)
        # results are rounded to 8 bits, half a step of 2^-8 at most; few of the query's
        # values the other way
        assert float((got.double() - exact).norm() / exact.norm()) < 2e-3
        assert not one._tickets.any()
        if captured:
            for c in (one, two):
                c.graph_pos += 1


def test_no_room():
    """A captured step behind the last place attends to what is there."""
    g = torch.Generator("cuda").manual_seed(3)
    one, two = _caches(2, 2, 64, 1024, 1024, True, g)
    (q, k, v), cos, sin = _token(2, 4, 2, 64, g)
    held = one._k.clone(), one._v.clone()
    got = one.attend_step(q, k, v, cos, sin, 0.1)
    qt = ops.apply_rope(q, cos, sin)
    last = torch.tensor([1023], dtype=torch.int32, device="cuda")
    want = ops.attention(qt.transpose(1, 2), two._k, two._v, 0.1, pos_dev=last)
    assert torch.equal(one._k, held[0]) and torch.equal(one._v, held[1])
    want = want.transpose(1, 2).reshape(2, 1, -1).float()
    assert float((got.float() - want).norm() / want.norm()) < 2e-3


def test_other_forms_are_left():
    g = torch.Generator("cuda").manual_seed(4)
    for Hq, Hkv, D in ((32, 1, 64), (4, 2, 96), (4, 2, 128)):
        (cache, _), ((q, k, v), cos, sin) = (_caches(1, Hkv, D, 8, 64, False, g),
                                             _token(1, Hq, Hkv, D, g))
        if D == 128:
            v = torch.cat([v, v], -1)[..., ::2]     # every second element
        assert cache.attend_step(q, k, v, cos, sin, 0.1) is None and cache.offset == 8


def test_replays():
    """A captured step, replayed at growing lengths among eager ones."""
    B, Hq, Hkv, D = 2, 8, 2, 128
    g = torch.Generator("cuda").manual_seed(5)
    one, two = _caches(B, Hkv, D, 120, 1000, True, g)
    (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
    for _ in range(2):
        one.attend_step(q, k, v, cos, sin, 0.1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = one.attend_step(q, k, v, cos, sin, 0.1)
    for step in range(12):
        graph.replay()
        qt, kt, vt = two.append_rope_qkv(q, k, v, cos, sin)
        want = ops.attention(qt.transpose(1, 2), kt, vt, 0.1, pos_dev=two.graph_pos)
        want = want.transpose(1, 2).reshape(B, 1, -1).float()
        assert float((got.float() - want).norm() / want.norm()) < 2e-3
        for c in (one, two):
            c.graph_pos += 7
            # the places in between are filled as a prompt would
            p = int(c.graph_pos)
            c._k[:, :, p - 6: p] = 0.5
            c._v[:, :, p - 6: p] = -0.5
        torch.cuda.synchronize()
    assert not one._tickets.any()


# partial results merged 4, 8 and 16 slices at once: fewer items than threads, a
# remainder, eight a thread; slices of a batch and one more
@pytest.mark.parametrize("B,Hq,Hkv,D,keys", [
    (1, 3, 1, 64, 200), (1, 3, 1, 64, 300), (1, 6, 2, 64, 1100), (1, 14, 2, 128, 250),
    (1, 14, 2, 128, 500), (2, 16, 1, 128, 257), (1, 32, 2, 128, 1500), (1, 16, 1, 256, 65),
    (1, 7, 1, 256, 300), (9, 16, 8, 256, 700)])
def test_merges(B, Hq, Hkv, D, keys):
    g = torch.Generator("cuda").manual_seed(keys)
    one, _ = _caches(B, Hkv, D, keys - 1, keys, False, g)
    (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
    got = one.attend_step(q, k, v, cos, sin, 0.1)
    exact = _exact(q, cos, sin, one.k, one.v, 0.0, 0)
    assert float((got.double() - exact).norm() / exact.norm()) < 2e-3  # as above
    assert not one._tickets.any()


@pytest.mark.parametrize("B,Hq,Hkv,D,keys,taken", [
    (1, 4, 1, 128, 8000, True), (1, 8, 1, 128, 2048, True), (1, 8, 1, 128, 2049, False),
    (1, 16, 1, 128, 1024, True), (1, 16, 1, 128, 1025, False), (1, 8, 8, 256, 1024, True),
    (1, 8, 8, 256, 1025, False), (1, 4, 4, 256, 100, False), (32, 8, 8, 256, 40, True),
    (33, 8, 8, 256, 40, False)])
def test_where_it_is_faster(B, Hq, Hkv, D, keys, taken):
    g = torch.Generator("cuda").manual_seed(keys)
    one, _ = _caches(B, Hkv, D, keys - 1, keys, False, g)
    (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
    got = one.attend_step(q, k, v, cos, sin, 0.1, faster=True)
    assert (got is not None) == taken and one.offset == (keys if taken else keys - 1)
    assert one.attend_step(q, k, v, cos, sin, 0.1) is not None


@pytest.mark.parametrize("B,Hq,Hkv,D,keys,window,taken", [
    (1, 8, 1, 128, 4000, 2048, True), (1, 8, 1, 128, 4000, 2049, False),
    (1, 4, 4, 256, 64, 0, True), (1, 4, 4, 256, 65, 0, False), (1, 4, 4, 256, 200, 64, True)])
def test_where_a_window_or_one_slice_is_faster(B, Hq, Hkv, D, keys, window, taken):
    g = torch.Generator("cuda").manual_seed(keys)
    one, _ = _caches(B, Hkv, D, keys - 1, keys, False, g)
    (q, k, v), cos, sin = _token(B, Hq, Hkv, D, g)
    got = one.attend_step(q, k, v, cos, sin, 0.1, window=window, faster=True)
    assert (got is not None) == taken
    if taken:
        exact = _exact(q, cos, sin, one.k, one.v, 0.0, window)
        assert float((got.double() - exact).norm() / exact.norm()) < 2e-3  # as above


# a wave's own tiles from 128 tiles of 64 keys of heads of 64 on, 512 of 128; before, and
# for heads of 256, tiles of a block
@pytest.mark.parametrize("B,Hq,Hkv,D,keys", [
    (4, 16, 4, 64, 448), (4, 16, 4, 64, 449), (16, 32, 8, 128, 192), (16, 32, 8, 128, 193),
    (64, 16, 8, 128, 64), (16, 8, 4, 256, 511)])
@pytest.mark.parametrize("window", [0, 100])
def test_attention_alone(B, Hq, Hkv, D, keys, window):
    g = torch.Generator("cuda").manual_seed(keys)
    new = lambda h, s: torch.randn(B, h, s, D, generator=g, device="cuda").bfloat16()  # noqa: E731
    q, k, v = new(Hq, 1), new(Hkv, keys), new(Hkv, keys)
    got = ops.attention(q, k, v, 0.1, sliding_window=window)
    one, zero = torch.ones(1, D // 2, device="cuda"), torch.zeros(1, D // 2, device="cuda")
    exact = _exact(q.transpose(1, 2), one, zero, k, v, 0.0, window)
    got = got.transpose(1, 2).reshape(B, 1, -1)
    assert float((got.double() - exact).norm() / exact.norm()) < 2e-3  # as above
