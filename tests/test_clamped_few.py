"""The clamped unit in the product of few rows."""

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


# both kernels of linear_own.hip, what linear_few.hip has of other units (four tiles a block of
# 32 and 64 rows), more rows than 64, ends of tiles, odd columns
@pytest.mark.parametrize("M,K,O", [
    (1, 96, 1), (16, 2048, 2304), (16, 544, 8200), (17, 96, 8192), (32, 1056, 8001), (33, 64, 8191),
    (64, 2048, 8192), (64, 160, 12000), (48, 992, 2049), (65, 512, 1000), (200, 2048, 2304)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("limit,alpha", [(7.0, 1.702), (0.5, 1.0)])
def test_unit(M, K, O, bias, limit, alpha):
    g = torch.Generator("cuda").manual_seed(M + O)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    x, w, b = rand(M, K), rand(2 * O, K) / K ** 0.5 * 3, rand(2 * O) if bias else None
    got = ops.clamped_few(x, w, b, limit, alpha)
    z = x.double() @ w.double().T
    # 32-bit sums
    off = (x.double().abs() @ w.double().abs().T) * (K * 2.0 ** -24)
    if bias:
        z = z + b.double()
        off = off + z.abs() * 2.0 ** -23
    gate, up = z.chunk(2, -1)
    gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    share = torch.sigmoid(alpha * gate)
    want = gate * share * (up + 1)
    # the unit of the gate grows by at most 1.13 of its argument; its exponential is off by
    # a few parts in 2^22
    og, ou = off.chunk(2, -1)
    off = 1.13 * og * ((up + 1).abs() + ou) + (gate * share).abs() * ou + want.abs() * 2.0 ** -20
    assert ((got.double() - want).abs() <= off + want.abs() * 2.0 ** -8 + 1e-6).all()


def test_apart():
    x = torch.randn(8, 512, device="cuda").bfloat16()
    w, b = torch.randn(256, 512, device="cuda").bfloat16(), torch.randn(256, device="cuda").bfloat16()
    assert ops.clamped_few(x, w, b, 7.0, 1.7) is not None
    for other in ((x.float(), w, b), (x, w.float(), b), (x, w, b[:128]), (x, w[:255], b[:255]),
                  (x, w, b.float()), (x[:, :256], w, b), (x.repeat(50, 1), w, b), (x.cpu(), w, b),
                  (x, w.t().contiguous().t(), b)):
        assert ops.clamped_few(*other, 7.0, 1.7) is None


# a few columns behind the biases' last, one and several tiles of them
@pytest.mark.parametrize("M,K,O,n", [(1, 96, 8, 1), (16, 544, 2304, 2300), (33, 64, 1024, 1017),
                                     (70, 512, 1000, 993)])
def test_biases_apart(M, K, O, n):
    g = torch.Generator("cuda").manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    x, w, pair = rand(M, K), rand(2 * O, K) / K ** 0.5, (rand(n), rand(n))
    both = torch.cat([torch.nn.functional.pad(b, (0, O - n)) for b in pair])
    assert torch.equal(ops.clamped_few(x, w, pair, 7.0, 1.7), ops.clamped_few(x, w, both, 7.0, 1.7))
    for other in ((pair[0], pair[1][:-1]), (pair[0], None), (pair[0], pair[1].float()),
                  (rand(O + 1), rand(O + 1)), (pair[0][:0], pair[1][:0]), (pair[0], pair[1].cpu())):
        assert ops.clamped_few(x, w, other, 7.0, 1.7) is None


@torch.no_grad()
@pytest.mark.parametrize("way", ["data", "parameter", "place"])
def test_replaced_biases(way):
    """Few rows have the biases that the module has now, as many rows have."""
    from mlx_sharding_amd.models.mixers import BiasedMLP
    from mlx_sharding_amd.ops.ragged import ClampedGLU
    torch.manual_seed(1)
    m = BiasedMLP(512, 300, ClampedGLU(7.0)).cuda()
    for p in m.parameters():
        p.data.normal_(0, 0.05)
    x = torch.randn(400, 512, device="cuda").bfloat16()
    before = m(x[:8])
    for part in (m.gate, m.up):
        new = torch.randn(300, device="cuda").bfloat16()
        if way == "data":
            part.bias.data = new
        elif way == "parameter":
            part.bias = torch.nn.Parameter(new, requires_grad=False)
        else:
            part.bias.copy_(new)
    few, many = m(x[:8]).double(), m(x)[:8].double()
    assert float((few - before.double()).norm() / few.norm()) > 0.1
    # many rows round the products and the unit to bf16 between
    assert float((few - many).norm() / many.norm()) < 4 * 2.0 ** -9
