"""Attention kernels at the edges of their tiles, against 64-bit attention."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def ext():
    from mlx_sharding_amd import ops
    e = ops.hip_ext()
    assert e is not None, "HIP extension must be built on a GPU box"
    return e


def attention(q, k, v, scale, cap, window, offset):
    """(output, what the weights' absolute values make of |v|) in 64 bits."""
    q, k, v = q.double(), k.double(), v.double()
    rep = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    if cap:
        s = torch.tanh(s / cap) * cap
    at = torch.arange(q.shape[2], device=q.device)[:, None] + offset
    key = torch.arange(k.shape[2], device=q.device)[None, :]
    hidden = key > at
    if window:
        hidden = hidden | (key <= at - window)
    p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
    return p @ v, p @ v.abs()


def cached(B, H, S, D, room):
    """Rows [B, H, S, D] of a cache whose other rows are NaN."""
    buf = torch.full((B, H, S + room, D), math.nan, dtype=torch.bfloat16,
                     device="cuda")
    buf[:, :, :S] = torch.randn(B, H, S, D, device="cuda")
    return buf[:, :, :S]


PREFILL = [(32, 16), (32, 32), (32, 64), (64, 32), (64, 64), (64, 128), (128, 32),
           (128, 64), (128, 128), (192, 64), (192, 128), (256, 256)]


@pytest.mark.parametrize("Dk,Dv", PREFILL)
def test_prefill_edges(Dk, Dv):
    """Tiles of 128 queries and 64 (32) keys: one query, one more and one less
    than a tile, windows that begin inside tiles, fewer heads than XCDs, a
    negative scale (and none), queries as slices of wider rows."""
    torch.manual_seed(Dk + Dv)
    for B, Hq, Hkv, T, offset, cap, window, scale in (
            (1, 8, 4, 1, 77, 0.0, 0, 0.1), (1, 4, 2, 57, 0, 0.0, 0, 0.1),
            (2, 8, 2, 129, 0, 0.0, 0, 0.1), (1, 2, 1, 127, 64, 20.0, 65, 0.1),
            (1, 3, 1, 300, 31, 30.0, 0, 0.2), (1, 8, 8, 130, 75, 0.0, 50, -0.1),
            (1, 2, 2, 33, 0, 0.0, 1, 0.1), (1, 2, 2, 128, 0, 0.0, 0, 0.0)):
        S = T + offset
        rows = torch.randn(B, T, Hq, Dk + 8, dtype=torch.bfloat16, device="cuda")
        q = rows[..., 8:].transpose(1, 2)
        k, v = cached(B, Hkv, S, Dk, 37), cached(B, Hkv, S, Dv, 37)
        out = ext().attn_prefill(q, k, v, scale, cap, window, offset).double()
        expect, size = attention(q, k, v, scale, cap, window, offset)
        # weights and result are rounded to bf16 (2^-8 each); exponents of up
        # to 2^8 in 32-bit steps come to less than 2^-13 of a weight
        bound = 2.0 ** -8 * (size + expect.abs()) + 2.0 ** -13 * size + 1e-6
        assert (out.shape == expect.shape
                and bool(((out - expect).abs() <= bound).all())), (T, offset, window)


def test_prefill_large_scores():
    """The reference of the exponents moves late and far: scores that grow
    with the key by hundreds, and one key that stands out."""
    torch.manual_seed(0)
    T, D = 200, 128
    q = torch.full((1, 8, T, D), 1.0, dtype=torch.bfloat16, device="cuda")
    k = (torch.arange(T, device="cuda") / D * 4).bfloat16()[None, None, :, None]
    k = k.expand(1, 8, T, D).contiguous()
    k[:, 1, 70] = 9.0
    v = torch.randn(1, 8, T, D, device="cuda").bfloat16()
    for scale in (1.0, 0.01, -1.0):
        out = ext().attn_prefill(q, k, v, scale, 0.0, 0, 0).double()
        expect, size = attention(q, k, v, scale, 0.0, 0, 0)
        # scores of up to 1200 are off by 2^-24 of themselves each way
        bound = 2.0 ** -8 * (size + expect.abs()) + 2.0 ** -12 * size + 1e-6
        assert bool(((out - expect).abs() <= bound).all()), scale


DECODE = [(4, 4, 64, 64), (8, 1, 64, 64), (8, 2, 128, 128), (14, 2, 128, 128),
          (12, 2, 128, 128), (16, 1, 128, 128), (3, 3, 192, 128),
          (16, 8, 256, 256), (16, 1, 576, 512), (4, 1, 576, 512)]


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("Hq,Hkv,Dk,Dv", DECODE)
def test_decode_edges(Hq, Hkv, Dk, Dv, captured):
    """Tiles of 64 or 32 keys and slices of them: one key, one more and one less
    than a tile, slices that are empty, windows that begin inside a tile; values
    within the keys' rows; the length on the device."""
    torch.manual_seed(Hq + Dk)
    for S in (1, 2, 31, 33, 64, 65, 500, 3001):
        for cap, window, scale in ((0.0, 0, 0.08), (30.0, 0, 0.1),
                                   (0.0, 100, -0.08), (50.0, 64, 0.2)):
            q = torch.randn(2, Hq, 1, Dk, dtype=torch.bfloat16, device="cuda") * 2
            k = cached(2, Hkv, S, Dk, 70)
            v = k[..., :Dv] if Dk == 576 else cached(2, Hkv, S, Dv, 70)
            given, pos = (k, v), None
            if captured:  # whole buffers and the last key's place
                given = [t.as_strided((2, Hkv, S + 70, t.shape[3]), t.stride())
                         for t in (k, v)]
                pos = torch.tensor([S - 1], dtype=torch.int32, device="cuda")
            out = ext().attn_decode(q, *given, scale, cap, window, pos).double()
            expect, size = attention(q, k, v, scale, cap, window, S - 1)
            # the result is rounded to bf16, exponents come in 32-bit steps
            bound = 2.0 ** -8 * expect.abs() + 2.0 ** -13 * size + 1e-6
            assert bool(((out - expect).abs() <= bound).all()), (S, cap, window)


@pytest.mark.parametrize("Hq,Hkv,Dk,Dv", [(8, 4, 128, 128), (8, 2, 64, 64)])
def test_heads_of_one_memory(Hq, Hkv, Dk, Dv):
    """Key and value heads that are one in memory, side by side in name only."""
    torch.manual_seed(3)
    q = torch.randn(1, Hq, 1, Dk, device="cuda").bfloat16()
    k, v = (cached(1, 1, 300, D, 10).expand(1, Hkv, 300, D) for D in (Dk, Dv))
    out = ext().attn_decode(q, k, v, 0.1, 0.0, 0, None).double()
    expect, size = attention(q, k, v, 0.1, 0.0, 0, 299)
    bound = 2.0 ** -8 * expect.abs() + 2.0 ** -13 * size + 1e-6
    assert bool(((out - expect).abs() <= bound).all())


def opposed(Hq, Hkv, Dk, Dv, S, step):
    """q, k, v whose values come in pairs of opposite sign, with scores (at a scale of
    1) that differ by twice ``step``: what is left of a pair's weights is their
    difference.  Scores lie in 32 bits as they are."""
    at = Dk - 2  # behind values that lie in the keys' rows
    q = torch.zeros(2, Hq, 1, Dk, device="cuda")
    q[..., at:] = 1.0
    k, v = cached(2, Hkv, S, Dk, 70), cached(2, Hkv, S, Dv, 70)
    base = torch.rand(2, Hkv, S // 2, device="cuda") - 1.0
    k[..., at] = base.repeat_interleave(2, 2).bfloat16()
    k[:, :, 0::2, at + 1], k[:, :, 1::2, at + 1] = step, -step
    if Dk == 576:
        v = k[..., :Dv]
    v[:, :, 1::2] = -v[:, :, 0::2]
    return q.bfloat16(), k, v


@pytest.mark.parametrize("Hq,Hkv,Dk,Dv", DECODE)
def test_decode_weights_are_whole(Hq, Hkv, Dk, Dv):
    """All 24 bits of the weights count."""
    torch.manual_seed(Hq + Dk)
    q, k, v = opposed(Hq, Hkv, Dk, Dv, 512, 2.0 ** -15)
    out = ext().attn_decode(q, k, v, 1.0, 0.0, 0, None).double()
    expect, _ = attention(q, k, v, 1.0, 0.0, 0, 511)
    # Of a difference of 2^-14: exponents in steps of 2^-24 and powers within 2^-23,
    # twice, make 2^-8.2 at most and less than half on average; the result is rounded
    # by 2^-9.  Weights of 16 bits would be off by 3%.
    assert (out - expect).norm() < 0.008 * expect.norm()


@pytest.mark.parametrize("cap", [5.0, 50.0])
def test_soft_cap_of_small_differences(cap):
    """Capped scores keep the bits of their differences."""
    torch.manual_seed(1)
    q, k, v = opposed(8, 2, 128, 128, 512, 2.0 ** -15)
    out = ext().attn_decode(q, k, v, 1.0, cap, 0, None).double()
    expect, _ = attention(q, k, v, 1.0, cap, 0, 511)
    # as above; the cap's own roundings are 2^-22 of scores of up to 1, twice.  Taken
    # from cap * (1 - 2 / (e^2y + 1)), scores were off by 2^-24 of the cap and more
    assert (out - expect).norm() < 0.012 * expect.norm()


@pytest.mark.parametrize("cap,scale", [(20.0, 1.0), (30.0, -0.5), (50.0, 3.0)])
def test_soft_cap_range(cap, scale):
    """Scores from far below the cap to far above it, of both signs, in waves that
    have only small ones and in mixed ones."""
    torch.manual_seed(2)
    D, S = 256, 300
    size = torch.logspace(-3, 1.3, S, device="cuda")[:, None]
    for top in (0.03, 1.0):
        k = (torch.randn(1, 2, S, D, device="cuda") * size * top).bfloat16()
        v = torch.randn(1, 2, S, D, device="cuda").bfloat16()
        q = torch.randn(1, 8, S, D, device="cuda").bfloat16() * 0.25
        for got, first in ((ext().attn_prefill(q, k, v, scale, cap, 0, 0), 0),
                           (ext().attn_decode(q[:, :, -1:], k, v, scale, cap, 0, None),
                            S - 1)):
            expect, whole = attention(q[:, :, first:], k, v, scale, cap, 0, first)
            # weights (of a prompt) and result are rounded to bf16; 32-bit scores
            # below the cap are off by 2^-21 of it, each way
            bound = (2.0 ** -8 * ((whole if first == 0 else 0) + expect.abs())
                     + cap * 2.0 ** -20 * whole + 1e-6)
            assert bool(((got.double() - expect).abs() <= bound).all()), (top, first)


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("N,S,nope,vdim", [(1, 1, 128, 128), (1, 3002, 128, 128),
                                           (3, 33, 32, 16), (17, 64, 160, 208),
                                           (64, 513, 128, 128), (129, 40, 64, 64)])
def test_latent_one_token(N, S, nope, vdim, captured):
    """One token per sequence over a cached latent, from projected rows to heads'
    outputs: remainders of 16 tokens, matrices of other sizes, one and many
    slices of the keys."""
    H, rank, rope, room = 16, 512, 64, 5
    torch.manual_seed(N + S)
    bf = lambda *s: torch.randn(*s, device="cuda").bfloat16()  # noqa: E731
    y = bf(N, H * (nope + rope) + rank + rope)
    q, latent = y.split([H * (nope + rope), rank + rope], -1)
    wk, wv = bf(H, rank, nope) * 0.1, bf(H, vdim, rank) * 0.05
    norm = (1 + 0.1 * torch.randn(rank, device="cuda")).bfloat16()
    angle = torch.rand(1, rope // 2, device="cuda") * 6
    cos, sin = torch.cos(angle), torch.sin(angle)
    cache = cached(N, 1, S - 1, rank + rope, room + 1).as_strided(
        (N, 1, S + room, rank + rope),
        ((S + room) * (rank + rope), (S + room) * (rank + rope), rank + rope, 1))
    before = cache.clone()
    pos = torch.tensor([S - 1], dtype=torch.int32, device="cuda")
    qf = ext().mla_prepare(q, latent, wk, norm, 1e-6, 0.0, cos, sin, cache,
                           pos if captured else None, 0 if captured else S - 1)
    out = ext().mla_attend(qf, cache, wv, 0.05, pos if captured else None,
                           1 if captured else S).double()

    def turned(t):
        a, b = t.double()[..., 0::2], t.double()[..., 1::2]
        c, s = cos.double(), sin.double()
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)

    close = lambda got, expect, off=0.0: bool(  # noqa: E731
        ((got.double() - expect).abs() <= 2.0 ** -8 * expect.abs() + off + 1e-5).all())
    # the token's row, and only that
    c = latent[:, :rank].double()
    row = torch.cat([c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + 1e-6)
                     * norm.double(), turned(latent[:, rank:])], -1)
    assert close(cache[:, 0, S - 1], row)
    cache_but = cache.clone()
    cache_but[:, 0, S - 1] = before[:, 0, S - 1]
    assert torch.equal(cache_but.view(torch.int16), before.view(torch.int16))
    # queries
    qh = q.reshape(N, H, nope + rope)
    heads_first = qh[..., :nope].double().transpose(0, 1).contiguous()
    space = torch.bmm(heads_first, wk.double().transpose(1, 2).contiguous())
    expect = torch.cat([space.transpose(0, 1), turned(qh[..., nope:])], -1)
    sums = torch.bmm(heads_first.abs(), wk.double().abs().transpose(1, 2).contiguous())
    assert close(qf[:, :, 0, :rank], expect[..., :rank],
                 sums.transpose(0, 1) * nope * 2.0 ** -24)
    assert close(qf[:, :, 0, rank:], expect[..., rank:])
    # outputs, from the queries and rows as they were rounded
    rows = cache[:, :, :S]
    o, size = attention(qf, rows, rows[..., :rank], 0.05, 0.0, 0, S - 1)
    o, size = (t[:, :, 0].transpose(0, 1).contiguous() for t in (o, size))
    w = wv.double().transpose(1, 2).contiguous()
    expect = torch.bmm(o, w).transpose(0, 1).reshape(N, -1)
    # the latents between the two products are rounded to bf16
    off = torch.bmm(2.0 ** -8 * o.abs() + 2.0 ** -13 * size, w.abs())
    assert close(out, expect, off.transpose(0, 1).reshape(N, -1))


@pytest.mark.parametrize("B,T,at,H", [(1, 2, 0, 2), (2, 33, 0, 3), (3, 130, 70, 16),
                                      (1, 300, 129, 8), (8, 128, 0, 16)])
def test_latent_prompt(B, T, at, H):
    """A prompt, or the next part of one, over keys in two parts: rows into the
    cache, then attention with queries that the kernel turns; tiles of 128 queries
    and 64 keys with remainders, operands as slices of wider rows."""
    rank, rope, room = 64, 64, 3
    S = at + T
    torch.manual_seed(S + H)
    bf = lambda *s: torch.randn(*s, device="cuda").bfloat16()  # noqa: E731
    q, latent = bf(B, T, H * 192 + rank + rope).split([H * 192, rank + rope], -1)
    norm = (1 + 0.1 * torch.randn(rank, device="cuda")).bfloat16()
    angle = torch.rand(T, rope // 2, device="cuda") * 6
    cos, sin = torch.cos(angle), torch.sin(angle)
    cache = cached(B, 1, at, rank + rope, room + T).as_strided(
        (B, 1, S + room, rank + rope),
        ((S + room) * (rank + rope), (S + room) * (rank + rope), rank + rope, 1))
    before = cache.clone()
    rows = ext().mla_rows(latent, norm, 1e-6, 0.0, cos, sin, cache, at, True)

    def turned(t, c, s):
        a, b = t.double()[..., 0::2], t.double()[..., 1::2]
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)

    close = lambda got, expect: bool(  # noqa: E731
        ((got.double() - expect).abs() <= 2.0 ** -8 * expect.abs() + 1e-5).all())
    c = latent[..., :rank].double()
    normed = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + 1e-6) * norm.double()
    assert close(rows, normed)
    new = cache[:, 0, at: S]
    assert torch.equal(new[..., :rank], rows)
    assert close(new[..., rank:], turned(latent[..., rank:], cos.double(), sin.double()))
    others = torch.cat([cache[:, :, :at], cache[:, :, S:]], 2)
    assert torch.equal(others.view(torch.int16),
                       torch.cat([before[:, :, :at], before[:, :, S:]], 2).view(torch.int16))
    kv = bf(B, S, H, 256)
    qh = q.view(B, T, H, 192)
    out = ext().mla_prompt(qh, kv, cache, cos, sin, 0.1, at).view(B, T, H, 128)
    k = torch.cat([kv[..., :128], cache[:, 0, :S, None, rank:].expand(B, S, H, 64)], -1)
    # queries are rounded behind their rotation
    qt = torch.cat([qh[..., :128].double(), turned(
        qh[..., 128:], cos.double()[:, None], sin.double()[:, None]).bfloat16().double()], -1)
    expect, size = attention(qt.transpose(1, 2), k.transpose(1, 2),
                             kv[..., 128:].transpose(1, 2), 0.1, 0.0, 0, at)
    # a query that rounds the other way than in 64 bits moves scores: 64 terms of
    # 2^-8 times |q k| near 1, few of them; weights are rounded to bf16
    bound = 2.0 ** -8 * expect.abs() + 2.0 ** -7 * size + 1e-5
    assert bool(((out.transpose(1, 2) - expect).abs() <= bound).all())


@pytest.mark.parametrize("Dk,Dv", [(32, 16), (64, 64), (128, 128), (192, 128), (256, 256)])
def test_prefill_two_teams(Dk, Dv):
    """Long keys of few blocks, whose tiles two teams take by turns: odd and even
    numbers of tiles, a team without a tile for a wave's queries, windows that begin
    inside either team's first tile, more blocks than CUs; scores that grow with the
    key and with its distance, so that either team's reference is far above."""
    torch.manual_seed(Dk + Dv)
    for B, Hq, Hkv, T, offset, cap, window, scale, slope in (
            (1, 8, 4, 641, 0, 0.0, 0, 0.1, 0), (1, 2, 1, 1, 704, 0.0, 0, 0.1, 0),
            (1, 4, 2, 130, 900, 20.0, 0, 0.1, 0), (2, 3, 1, 200, 1000, 0.0, 700, 0.1, 0),
            (1, 2, 2, 64, 2000, 0.0, 737, -0.1, 0), (1, 24, 8, 1600, 0, 0.0, 0, 0.1, 0),
            (1, 2, 2, 150, 600, 0.0, 0, 1.0, 4), (1, 2, 2, 150, 600, 0.0, 0, 1.0, -4)):
        S = T + offset
        q = torch.randn(B, Hq, T, Dk, device="cuda").bfloat16()
        k, v = cached(B, Hkv, S, Dk, 37), cached(B, Hkv, S, Dv, 37)
        if slope:
            q[..., 0] = 1.0
            k[..., 0] = torch.arange(S, device="cuda") / 4 * slope
        out = ext().attn_prefill(q, k, v, scale, cap, window, offset).double()
        expect, size = attention(q, k, v, scale, cap, window, offset)
        # as above; scores of up to 800 are off by 2^-24 of themselves each way
        bound = 2.0 ** -8 * (size + expect.abs()) + 2.0 ** -12 * size + 1e-6
        assert (out.shape == expect.shape
                and bool(((out - expect).abs() <= bound).all())), (T, offset, window, slope)


@pytest.mark.parametrize("B,T,at,H", [(1, 700, 0, 2), (2, 129, 640, 3)])
def test_latent_prompt_two_teams(B, T, at, H):
    test_latent_prompt(B, T, at, H)
