"""Products of few rows: every number of tiles a block that their sizes lead to, ragged ends."""

import types

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


def check(M, K, O, act, norm, bias, residual):
    g = torch.Generator("cuda").manual_seed(O + M + K)

    def rand(*n):
        return torch.randn(*n, generator=g, device="cuda").bfloat16()

    rows = 2 * O if act else O
    x, w = rand(M, K), rand(rows, K) / K ** 0.5
    n = types.SimpleNamespace(weight=rand(K), eps=1e-5, weight_offset=0.5) if norm else None
    b = rand(rows) if bias else None
    res = rand(M, O) if residual else None
    h = x.double()
    if norm:
        h = (h * (h.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
             * (n.weight.double() + 0.5))
    z = h @ w.double().T
    # 32-bit sums, and rows rounded to bf16 behind the norm
    off = (h.abs() @ w.double().abs().T) * (K * 2.0 ** -24 + (2.0 ** -8 if norm else 0.0))
    if bias:
        z = z + b.double()
        off = off + z.abs() * 2.0 ** -23
    if act:  # either unit grows by at most 1.13 of its argument
        gate, up, og, ou = *z.chunk(2, -1), *off.chunk(2, -1)
        unit = (torch.nn.functional.silu(gate) if act == "silu" else
                torch.nn.functional.gelu(gate, approximate="tanh"))
        z, off = unit * up, 1.13 * og * (up.abs() + ou) + unit.abs() * ou + 1e-6
    if residual:
        z = z + res.double()
    got = ops._linear_few(x, w, b, res, n, act)
    assert got is not None
    # the result is rounded to bf16
    assert ((got.double() - z).abs() <= off + z.abs() * 2.0 ** -8 + 1e-6).all()


# tiles of 16 rows of W (8 columns of a unit) at both ends of the ranges that have one to eight
# tiles a block
@pytest.mark.parametrize("act", [None, "silu"])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("M,K", [(1, 96), (16, 1120), (17, 160), (32, 64), (33, 96), (64, 1056)])
@pytest.mark.parametrize("tiles", [1, 128, 129, 256, 257, 384, 385, 512, 513, 768, 769, 1024,
                                   1025, 1280, 1281, 1536, 1537, 1792, 1793, 2048,
                                   2049])
def test_tiles(M, K, tiles, norm, act):
    check(M, K, tiles * (8 if act else 16) - 4, act, norm, not norm, norm == bool(act))


# sums of three columns at the end, odd ones, one; contractions of one step and of parts of a
# chunk, a stage and a round of the waves
@pytest.mark.parametrize("act", [None, "silu", "gelu_tanh"])
@pytest.mark.parametrize("M", [2, 15, 18, 31, 47, 63])
@pytest.mark.parametrize("O,K", [(1, 32), (13, 992), (2049, 32), (4110, 544), (9001, 96),
                                 (15001, 224), (300, 8192)])
def test_ends(M, O, K, act):
    check(M, K, O, act, True, False, False)
    check(M, K, O, act, False, True, True)


# long contractions into many columns
@pytest.mark.parametrize("act", [None, "silu"])
@pytest.mark.parametrize("M,K,O", [(9, 8224, 4097), (17, 9216, 8200), (64, 8224, 4112),
                                   (33, 16352, 5000), (64, 13824, 9001)])
def test_long(M, K, O, act):
    check(M, K, O, act, False, True, True)
    check(M, K, O, act, True, False, False)


# 65 and more rows: groups of 32 and 64, with as many tiles as fit a round of 256 blocks, and one
# more; the longest contraction, and the shortest
@pytest.mark.parametrize("act", [None, "silu", "gelu_tanh"])
@pytest.mark.parametrize("M,K", [(65, 512), (96, 1056), (97, 544), (128, 8192), (129, 608), (192, 992),
                                 (384, 576)])
@pytest.mark.parametrize("of,rt", [(32, 1), (32, 2), (32, 3), (64, 1), (64, 2), (64, 3), (64, 4),
                                   (64, 5), (64, 6), (64, 8)])
def test_more_rows(M, K, of, rt, act):
    if rt > 5 and M > 128:
        return
    tiles = rt * (256 // (-(-M // of)))
    for t in (tiles - rt + 1, tiles):
        check(M, K, t * (8 if act else 16) - 3, act, False, rt % 2 == 0, False)


# contractions that two and four blocks share, from the shortest on, with ends of tiles, chunks
# and shares
@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("I,O", [(5632, 2048), (5664, 1040), (5696, 1024), (6176, 3), (16384, 900)])
def test_shared(M, I, O):
    g = torch.Generator("cuda").manual_seed(I + O)

    def rand(*n):
        return torch.randn(*n, generator=g, device="cuda").bfloat16()

    x, w_in, w_out = rand(M, 64), rand(2 * I, 64) / 8, rand(O, I) / I ** 0.5
    res = rand(M, O)
    for _ in range(3):  # numbers are cleared each time
        got = ops.feed_few(x, w_in, w_out, "silu", None, res)
        units = ops._linear_few(x, w_in, None, None, None, "silu")
        want = units.double() @ w_out.double().T + res.double()
        off = (units.double().abs() @ w_out.double().abs().T) * (I * 2.0 ** -24)
        assert ((got.double() - want).abs() <= off + want.abs() * 2.0 ** -8 + 1e-6).all()
