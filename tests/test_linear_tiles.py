"""Products of more than 64 rows on the experts' tiles, against 64 bits."""

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu

ACTS = {0: None, 1: "silu", 2: "gelu_tanh"}


def ext():
    e = ops.hip_ext()
    assert e is not None, "HIP extension must be built on a GPU box"
    return e


def operands(M, O, K, wide=0):
    g = torch.Generator().manual_seed(M + O + K)
    new = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x = new(M, K + wide).bfloat16().cuda()[:, wide:]
    w = (new(O, K + wide) * 0.05).bfloat16().cuda()[:, :K]
    return x, w, new(O).bfloat16().cuda()


def exact(x, w, bias, act):
    """(result in 64 bits, how far sums of 32 bits and a result in bf16 may be off)."""
    z = x.double() @ w.double().T
    off = (x.double().abs() @ w.double().abs().T) * w.shape[1] * 2.0 ** -24
    if bias is not None:
        z = z + bias.double()
    if act:
        gate, up = z.chunk(2, -1)
        og, ou = off.chunk(2, -1)
        unit = F.silu if act == 1 else lambda t: F.gelu(t, approximate="tanh")
        z = unit(gate) * up
        # a unit's slope is below 1.13; its exponential and quotient are 32 bits wide
        off = 1.13 * og * up.abs() + unit(gate).abs() * ou + 2.0 ** -20 * z.abs()
    return z, off + 2.0 ** -8 * z.abs() + 1e-30


# one row, tiles' edges and one row more, two tiles and a remainder; remainders of 256 and
# of 128 columns; three stages (as many as there are places), four, and more; several
# items a block; shares of unequal length
@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("M,O,K", [
    (1, 64, 192), (65, 128, 256), (128, 320, 192), (129, 256, 448), (256, 192, 320),
    (257, 1088, 1024), (300, 576, 704), (2100, 4160, 192), (1100, 8192, 256)])
def test_against_64_bits(M, O, K, tile):
    x, w, bias = operands(M, O, K, wide=8 if K % 128 else 0)
    for act in (0, 1, 2):
        if O % (128 if act else 64):
            continue
        for b in ((None, bias) if not act else (None,)):
            for shares in (1, 2, 3, 5):
                if K // 64 // shares < 3 or (act and shares > 1):
                    continue
                got = ext().linear_tiles(x, w, b, act, tile, shares).double()
                want, off = exact(x, w, b, act)
                assert bool(((got - want).abs() <= off).all()), (act, shares)


def test_refusals():
    x, w, bias = operands(100, 128, 512)
    for args in ((x[:, :448], w, None, 0, 128, 1), (x, w, None, 0, 64, 1),
                 (x, w, None, 1, 128, 2), (x, w, bias, 1, 128, 1), (x, w, None, 3, 128, 1),
                 (x, w, None, 0, 128, 3), (x, w[:96], None, 0, 128, 1),
                 (x.float(), w.float(), None, 0, 128, 1), (x, w, bias[:64], 0, 128, 1),
                 (x.cpu(), w, None, 0, 128, 1), (x, w, None, 0, 128, 0)):
        with pytest.raises(RuntimeError):
            ext().linear_tiles(*args)


@pytest.mark.parametrize("M,O,K,act", [
    (65, 1024, 8192, 0), (300, 1536, 8960, 0), (1280, 1024, 8192, 0),
    (2000, 5632, 2048, 1), (1400, 4096, 1024, 2)])
def test_forms_that_the_rule_takes(M, O, K, act):
    """Batches of sequences, slices of wider ones, biases: taken or not, they are what
    separate operators give."""
    x, w, bias = operands(M, O, K)
    assert ext().linear_tiles_plan(M, O // (2 if act else 1), K, act, False)[0]
    # (a view in two dimensions more, rows of a wider one, rows off 16 bytes)
    forms = [x, x.view(M, 1, K) if M % 2 else x.view(2, M // 2, K),
             torch.cat([x, x], 1)[:, :K],
             torch.cat([x[:, :1], x, x[:, :1]], 1)[:, 1:K + 1]]
    for t in forms:
        for b in (None, bias, bias[:1].expand(O)):
            want, off = exact(t.reshape(M, K), w, b, act)
            got = ops.project(t, w, b, act=ACTS[act])
            assert got.shape == (*t.shape[:-1], want.shape[-1])
            if act:
                # apart, both halves are rounded to bf16 before the unit, and before a
                # bias in a form of its own
                z = exact(t.reshape(M, K), w, b, 0)[0].abs()
                if b is not None:
                    z = z + b.double().abs()
                gate, up = z.chunk(2, -1)
                off = off + 2.0 ** -7 * 1.13 * gate * up * (1 if b is None else 2)
            elif b is not None:
                off = off + 2.0 ** -8 * (want.abs() + b.double().abs())
            assert bool(((got.reshape(M, -1).double() - want).abs() <= off).all())


@pytest.mark.parametrize("M,O,K,taken", [
    (65, 1024, 8128, False), (65, 1024, 8192, True), (65, 960, 8192, False),
    (65, 1600, 8192, True), (65, 1664, 8192, False), (2560, 1024, 8192, True),
    (2561, 1024, 8192, False), (65, 1984, 10176, True), (65, 2048, 10176, False),
    (65, 5120, 10240, True), (65, 5184, 10240, False), (5120, 1024, 12288, True),
    (5121, 1024, 12288, False), (2048, 4096, 14336, True), (2049, 4096, 14336, False),
    (1905, 3584, 14336, True), (65, 5440, 16384, True), (65, 5504, 16384, False),
    (64, 3584, 14336, False)])
def test_borders_of_the_rule_for_long_contractions(M, O, K, taken):
    assert bool(ext().linear_tiles_plan(M, O, K, 0, False)[0]) == taken


def test_what_is_watched_keeps_torch():
    x, w, _ = operands(300, 1024, 8192)
    assert ops._linear_few(x, w) is not None
    p = torch.nn.Parameter(w.clone())
    assert ops._linear_few(x, p) is None
    ops.linear(x, p).float().sum().backward()
    assert p.grad is not None
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        assert torch.autograd.forward_ad.unpack_dual(ops.linear(dual, w)).tangent is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    want, off = exact(x, w, None, 0)
    mapped = torch.vmap(lambda r: ops.linear(r, w))(x.view(3, 100, 8192))
    assert bool(((mapped.reshape(300, -1).double() - want).abs() <= off).all())


def test_captured_and_replayed():
    """Shares' sums are the graph's own memory, and a replay reads what is there then."""
    x, w, _ = operands(200, 1024, 8192)
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.linear(x, w)
    torch.cuda.current_stream().wait_stream(s)
    with torch.cuda.graph(g):
        y = ops.linear(x, w)
    for k in range(3):
        x.copy_(torch.randn_like(x) * (k + 1))
        g.replay()
        eager = ops.linear(x, w)
        torch.cuda.synchronize()
        assert torch.equal(y, eager)
