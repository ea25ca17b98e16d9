"""Routed experts of a prompt on tiles of one expert, against 64-bit products."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def ext():
    from mlx_sharding_amd import ops
    e = ops.hip_ext()
    assert e is not None, "HIP extension must be built on a GPU box"
    return e


def routes(kind, N, E, top, gen):
    if kind == "one":       # every pair at one expert, the others have none
        return torch.full((N, top), E - 1, device="cuda")
    if kind == "few":       # experts without pairs in between
        return 2 * torch.randint(0, (E + 1) // 2, (N, top), generator=gen, device="cuda")
    return torch.rand(N, E, generator=gen, device="cuda").topk(top).indices


# one stage more than the ring has, remainders of the tiles of 256 and 128 rows of
# weights, tiles of one pair, as many pairs as a tile has and one more, many tiles a
# block, with two, three and more stages of 64 columns; more than one placing block
@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("N,E,top,H,I,kind", [
    (1, 3, 1, 128, 128, "any"), (257, 3, 1, 192, 320, "one"), (256, 2, 1, 128, 192, "one"),
    (43, 8, 6, 128, 192, "any"), (700, 7, 3, 320, 128, "few"), (1500, 160, 6, 256, 448, "any"),
    (5000, 4, 2, 512, 704, "any"), (3000, 160, 6, 1024, 128, "any"),
    (2000, 160, 6, 1088, 192, "any"), (1500, 160, 6, 128, 1024, "any")])
def test_against_64_bits(N, E, top, H, I, kind, tile):
    gen = torch.Generator("cuda").manual_seed(N + H)
    bf = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    x = bf(N, H + 8)[:, 8:] * 0.5  # rows of a wider one
    x = torch.empty(N, H + 8, dtype=torch.bfloat16, device="cuda")[:, :H].copy_(x)
    gate, up, down = bf(E, I, H) * 0.1, bf(E, I, H) * 0.1, bf(E, H, I) * 0.1
    choice = routes(kind, N, E, top, gen)
    y, where = ext().moe_tiles(x, choice, gate, up, down, tile)
    flat = where.flatten().long()
    assert torch.equal(flat.sort().values, torch.arange(N * top, device="cuda"))
    e = torch.empty(N * top, dtype=torch.long, device="cuda")
    e[flat] = choice.flatten()
    assert bool((e[1:] >= e[:-1]).all())
    for n in range(E):
        at = (choice.flatten() == n).nonzero().flatten()
        if not len(at):
            continue
        xe = x[at // top].double()
        g = xe @ gate[n].double().T
        h = torch.nn.functional.silu(g) * (xe @ up[n].double().T)
        expect = h @ down[n].double().T
        # h and y are rounded to bf16, sums are 32 bits wide
        bound = 2.0 ** -8 * (expect.abs() + h.abs() @ down[n].double().abs().T) + 1e-5
        assert bool(((y[flat[at]].double() - expect).abs() <= bound).all()), n


def test_other_sizes_take_the_general_path():
    """The rule's two sides give the same layer: widths that are no multiple of 64,
    and weights that somebody differentiates, go on as before."""
    from mlx_sharding_amd import ops
    gen = torch.Generator("cuda").manual_seed(1)
    bf = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    N, E, top, H, I = 300, 4, 2, 256, 192
    x, stacks = bf(N, H) * 0.5, [bf(E, I, H) * 0.1, bf(E, I, H) * 0.1, bf(E, H, I) * 0.1]
    w, choice = torch.rand(N, E, generator=gen, device="cuda").softmax(-1).topk(top)
    assert ops._tiles_ok(x, *stacks)
    tiles = ops.grouped_expert_mlp(x, *stacks, w, choice)
    tracked = [s.clone().requires_grad_() for s in stacks]
    assert not ops._tiles_ok(x, *tracked)
    general = ops.grouped_expert_mlp(x, *tracked, w, choice)
    # gate, up, unit and output are rounded to bf16 there
    scale = general.float().abs().max()
    assert (tiles.float() - general.detach().float()).abs().max() <= 2.0 ** -5 * scale
    one = x[:1].expand(N, H)  # one row in memory
    many = ops.grouped_expert_mlp(one, *stacks, w, choice)
    expect = ops.grouped_expert_mlp(one.contiguous(), *stacks, w, choice).float()
    assert (many.float() - expect).abs().max() <= 2.0 ** -5 * expect.abs().max()
    odd = [s[:, :100].contiguous() for s in stacks[:2]] + [stacks[2][..., :100].contiguous()]
    assert not ops._tiles_ok(x, *odd)
    assert ops.grouped_expert_mlp(x, *odd, w, choice).shape == (N, H)
