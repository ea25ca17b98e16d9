"""Routed experts of a decoding step: uneven choices, and a shared feed-forward beside."""

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops
from test_moe_rows import stack

pytestmark = pytest.mark.gpu


def _exact(y, choice, weight, gd, ud, dd):
    out = y.new_zeros(*choice.shape, dd.shape[1], dtype=torch.float64)
    a = y.double()
    for e in range(gd.shape[0]):
        t, k = (choice == e).nonzero(as_tuple=True)
        unit = F.silu(a[t] @ gd[e].T) * (a[t] @ ud[e].T)
        out[t, k] = weight[t, k, None].double() * (unit @ dd[e].T)
    return out.flatten(0, 1)


@pytest.mark.parametrize("N,E,top,I,H,bits", [
    (1, 64, 6, 128, 256, 4), (128, 64, 8, 128, 256, 4), (40, 64, 2, 256, 512, 16),
    (17, 2, 1, 1408, 2048, 8), (128, 5, 1, 128, 128, 4), (33, 64, 1, 384, 1024, 4)])
@pytest.mark.parametrize("uneven", ["all the same", "one of many", "random", "last"])
def test_shares(N, E, top, I, H, bits, uneven):
    """Blocks share the tiles of however many pairs an expert has."""
    gen = torch.Generator("cuda").manual_seed(N + E)
    (g, gd), (u, ud) = stack(E, I, H, bits, 64, gen), stack(E, I, H, bits, 64, gen)
    d, dd = stack(E, H, I, bits, 64, gen)
    y = torch.randn(N, H, generator=gen, device="cuda").bfloat16()
    choice = torch.stack([torch.randperm(E, generator=gen, device="cuda")[:top]
                          for _ in range(N)])
    if uneven == "all the same":
        choice[:] = torch.arange(top, device="cuda")
    elif uneven == "last":
        choice[:] = E - 1 - torch.arange(top, device="cuda")
    elif uneven == "one of many":
        choice[:, 0] = E // 2
        for row in choice:
            others = torch.randperm(E - 1, generator=gen, device="cuda")[: top - 1]
            row[1:] = (E // 2 + 1 + others) % E
    choice = choice.int().contiguous()
    weight = torch.rand(N, top, generator=gen, device="cuda")
    got = ops.expert_rows(y, choice, weight, g, u, d, bits, 64).double()
    want = _exact(y, choice, weight, gd, ud, dd)
    # fp16 weights and units (2^-12 each in the mean), bf16 units otherwise (2^-9)
    assert float((got - want).norm() / want.norm()) < (4e-3 if bits == 16 else 1e-3)


@pytest.mark.parametrize("N", [1, 7, 8])
@pytest.mark.parametrize("S,bits,H", [
    (64, 4, 512), (576, 16, 512), (4096, 4, 512),
    (4096, 4, 4096)])    # 256 blocks beside, of kernels of which a CU has one block
def test_shared_beside(N, S, bits, H):
    E, top, I = 16, 3, 128
    gen = torch.Generator("cuda").manual_seed(N + S)
    randn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    g, u = stack(E, I, H, bits, 64, gen)[0], stack(E, I, H, bits, 64, gen)[0]
    d = stack(E, H, I, bits, 64, gen)[0]
    w_in = (randn(2 * S, H) * H ** -0.5).bfloat16()
    w_out = (randn(H, S) * S ** -0.5).bfloat16()
    y = randn(N, H).bfloat16()
    choice = torch.stack([torch.randperm(E, generator=gen, device="cuda")[:top]
                          for _ in range(N)]).int()
    weight = torch.rand(N, top, generator=gen, device="cuda")
    assert ops.expert_shared_ok(N, H, w_in, w_out)
    rows, shared = ops.expert_rows(y, choice, weight, g, u, d, bits, 64, (w_in, w_out))
    assert torch.equal(rows, ops.expert_rows(y, choice, weight, g, u, d, bits, 64))
    a, b = (y.double() @ w_in.double().T).chunk(2, -1)
    want = (F.silu(a) * b) @ w_out.double().T
    # units and rows are rounded to bf16
    assert float((shared.double() - want).norm() / want.norm()) < 4e-3


def test_shared_apart():
    """What the kernels beside do not take."""
    w = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    assert not ops.expert_shared_ok(9, 512, w(256, 512), w(512, 128))
    assert not ops.expert_shared_ok(1, 512, w(192, 512), w(512, 96))
    assert not ops.expert_shared_ok(1, 512, w(2 * 4160, 512), w(512, 4160))
    assert not ops.expert_shared_ok(1, 512, w(256, 512), None)
    assert not ops.expert_shared_ok(1, 512, w(256, 520)[:, :512], w(512, 128))


# up to 64 pairs by ballots, more by counts: both sides of the line, groups of one expert
# that fill up, shares that end with a group (rows a multiple of them) and that do not,
# blocks with nothing to do
@pytest.mark.parametrize("N,E,top,I,H,bits", [
    (64, 3, 1, 128, 384, 4), (65, 3, 1, 128, 384, 4), (32, 64, 2, 384, 640, 8),
    (33, 64, 2, 384, 640, 8), (16, 64, 4, 1408, 512, 4), (10, 64, 6, 128, 3072, 16),
    (3, 64, 1, 128, 5120, 4)])
@pytest.mark.parametrize("spread", [1, 5, 64])
def test_groups(N, E, top, I, H, bits, spread):
    gen = torch.Generator("cuda").manual_seed(N + I)
    (g, gd), (u, ud) = stack(E, I, H, bits, 64, gen), stack(E, I, H, bits, 64, gen)
    d, dd = stack(E, H, I, bits, 64, gen)
    y = torch.randn(N, H, generator=gen, device="cuda").bfloat16()
    # pairs at the last few experts
    few = max(top, min(E, spread))
    choice = E - 1 - torch.stack([torch.randperm(few, generator=gen, device="cuda")[:top]
                                  for _ in range(N)])
    choice = choice.int().contiguous()
    weight = torch.rand(N, top, generator=gen, device="cuda")
    got = ops.expert_rows(y, choice, weight, g, u, d, bits, 64).double()
    want = _exact(y, choice, weight, gd, ud, dd)
    # as above
    assert float((got - want).norm() / want.norm()) < (4e-3 if bits == 16 else 1e-3)
