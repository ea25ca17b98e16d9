"""What few rows' products add to their columns, read by fours or alone."""

import types

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", [None, "silu"])
@pytest.mark.parametrize("M,O,K", [(1, 4, 32), (3, 20, 96), (16, 68, 64), (5, 8196, 160),
                                   (17, 4, 32), (33, 4100, 96), (64, 36, 2080),
                                   (2, 70, 64), (40, 18, 64)])
@pytest.mark.parametrize("shift,pad", [(0, 0), (1, 0), (0, 3), (4, 8)])
def test_ends(M, O, K, act, shift, pad):
    g = torch.Generator("cuda").manual_seed(O + M)

    def rand(*n):
        return torch.randn(*n, generator=g, device="cuda").bfloat16()

    rows = 2 * O if act else O
    x, w = rand(M, K), rand(rows, K) / K ** 0.5
    bias = rand(rows + 8)[shift: shift + rows]
    res = rand(M * (O + pad) + 8)[shift: shift + M * (O + pad)].view(M, O + pad)[:, :O]
    z = x.double() @ w.double().T + bias.double()
    if act:
        z = torch.nn.functional.silu(z[:, :O]) * z[:, O:]
    want = z + res.double()
    got = ops._linear_few(x, w, bias, res, None, act)
    # half a place of bf16, and sums of K products in fp32
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=1e-4)


# where a round of 256 blocks ends, for each number of tiles, and where rows of x change
# between registers and LDS
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("act", [None, "silu"])
@pytest.mark.parametrize("M,K", [(1, 64), (8, 4096), (9, 2048), (16, 2016), (17, 96), (64, 64)])
@pytest.mark.parametrize("rows", [4096, 4112, 8192, 8224, 12304, 16416, 24608])
def test_rounds(M, K, rows, act, norm):
    g = torch.Generator("cuda").manual_seed(rows + M)

    def rand(*n):
        return torch.randn(*n, generator=g, device="cuda").bfloat16()

    x, w = rand(M, K), rand(rows, K) / K ** 0.5
    n = types.SimpleNamespace(weight=rand(K), eps=1e-5, weight_offset=0.0) if norm else None
    h = x.double()
    if norm:
        h = h * (h.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * n.weight.double()
    z = h @ w.double().T
    # 32-bit sums, and rows rounded to bf16 behind the norm
    off = (h.abs() @ w.double().abs().T) * (K * 2.0 ** -24 + (2.0 ** -8 if norm else 0.0))
    if act:  # silu grows by at most 1.13 of its argument
        gate, up, og, ou = *z.chunk(2, -1), *off.chunk(2, -1)
        unit = torch.nn.functional.silu(gate)
        z, off = unit * up, 1.13 * og * (up.abs() + ou) + unit.abs() * ou + 1e-6
    got = ops._linear_few(x, w, None, None, n, act)
    assert bool(((got.double() - z).abs() <= 2.0 ** -8 * z.abs() + off + 1e-6).all())


# rows of W that lie a multiple of 2048 apart: blocks begin at columns of their own and go
# round, through registers and LDS, with fewer chunks than blocks and an incomplete last one
@pytest.mark.parametrize("M", [3, 12, 40])
@pytest.mark.parametrize("O,K", [(48, 2048), (4500, 96), (4500, 2016), (9000, 160), (9000, 2048)])
@pytest.mark.parametrize("act", [None, "silu"])
def test_rows_apart(M, O, K, act):
    g = torch.Generator("cuda").manual_seed(O + M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(2 * O if act else O, 2048, generator=g, device="cuda") / K ** 0.5
         ).bfloat16()[:, :K]
    z = x.double() @ w.double().T
    if act:
        z = torch.nn.functional.silu(z[:, :O]) * z[:, O:]
    got = ops._linear_few(x, w, None, None, None, act)
    # half a place of bf16, and sums of K products in fp32
    torch.testing.assert_close(got.double(), z, rtol=2 ** -8, atol=1e-4)
