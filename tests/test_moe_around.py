"""Halves of a shared feed-forward with the router and with the sum of a decoding step."""

import types

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops
from mlx_sharding_amd.models.fuse import fuse_model
from test_moe_rows import decoder_layer

pytestmark = pytest.mark.gpu


def fused_layer(bits):
    """One whose shared experts have their two first matrices side by side."""
    layer = decoder_layer(bits)
    fuse_model(layer)
    assert layer.mlp.shared_experts._fused_gu is not None
    return layer


# one block of tokens and two, groups of 16, 32 and 64 rows and one more; parts of 16 experts;
# every number of tiles a block, with a last one that is not whole
@pytest.mark.parametrize("N", [1, 7, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("E,top,H,S", [
    (64, 6, 2048, 2816), (1, 1, 128, 64), (17, 2, 4096, 8192), (48, 8, 2176, 4160),
    (33, 33, 640, 1088)])
def test_around(N, E, top, H, S):
    g = torch.Generator("cuda").manual_seed(N + E)
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x = randn(N, H).bfloat16()
    norm = types.SimpleNamespace(weight=(1 + 0.1 * randn(H)).bfloat16(), eps=1e-6,
                                 weight_offset=0.5)
    router = (randn(E, H) * 0.05).bfloat16()
    w_in = (randn(2 * S, H) * H ** -0.5).bfloat16()
    w_out = (randn(H, S) * S ** -0.5).bfloat16()
    assert ops.expert_begin_ok(N, H, w_in, w_out)
    zeros = lambda: torch.zeros(N, dtype=torch.int32, device="cuda")  # noqa: E731
    y, h, choice, weight, units = ops.expert_route(x, None, norm, router, top, 1.5, True,
                                                   zeros(), w_in)
    one = ops.expert_route(x, None, norm, router, top, 1.5, True)
    assert torch.equal(h, x)
    # sums of squares and products have other orders, as in test_route_parts
    assert torch.allclose(one[0].float(), y.float(), rtol=2.0 ** -7, atol=1e-6)
    p = torch.softmax(y.double() @ router.double().T, -1)
    own = p.gather(1, choice.long())
    assert bool((choice.sort(-1).values.diff(dim=-1) > 0).all())
    assert bool(((own - p.topk(top, -1).values).abs() <= 1e-5).all())
    assert bool(((weight.double() - 1.5 * own / own.sum(-1, keepdim=True)).abs() <= 1e-5).all())

    a = x.double()
    a = a * (a.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (norm.weight.double() + 0.5)
    z = a @ w_in.double().T
    # 32-bit sums of rows rounded to bf16; a unit grows by at most 1.13 of its argument
    off = (a.abs() @ w_in.double().abs().T) * (H * 2.0 ** -24 + 2.0 ** -8)
    gate, up, og, ou = *z.chunk(2, -1), *off.chunk(2, -1)
    want = F.silu(gate) * up
    off = 1.13 * og * (up.abs() + ou) + F.silu(gate).abs() * ou + want.abs() * 2.0 ** -8
    assert bool(((units.double() - want).abs() <= off + 1e-6).all())

    rows = randn(N * top, H)
    out = ops.expert_finish(units, w_out, rows, h).double()
    u, wd = units.double(), w_out.double()
    want = u @ wd.T + rows.double().view(N, top, H).sum(1) + x.double()
    off = ((u.abs() @ wd.abs().T + rows.double().abs().view(N, top, H).sum(1) + x.double().abs())
           * ((S + top) * 2.0 ** -24) + want.abs() * 2.0 ** -8)
    assert bool(((out - want).abs() <= off + 1e-6).all())


def test_apart():
    """What the two do not take."""
    w = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    assert not ops.expert_begin_ok(65, 512, w(256, 512), w(512, 128))
    assert not ops.expert_begin_ok(1, 4224, w(256, 4224), w(4224, 128))
    assert not ops.expert_begin_ok(1, 512, w(192, 512), w(512, 96))
    assert not ops.expert_begin_ok(1, 512, None, w(512, 128))
    assert not ops.expert_begin_ok(1, 512, w(256, 520)[:, :512], w(512, 128))
    assert not ops.expert_begin_ok(1, 512, w(256, 512).float(), w(512, 128))
    norm = types.SimpleNamespace(weight=w(128), eps=1e-6, weight_offset=0.0)
    for n, res in ((None, None), (2, w(2, 128))):
        with pytest.raises(RuntimeError):
            ops.expert_route(w(2, 128), res, norm, w(4, 128), 1, 1.0, False,
                             n and torch.zeros(n, dtype=torch.int32, device="cuda"), w(128, 128))


@pytest.mark.parametrize("bits,B,taken", [(0, 1, False), (4, 8, False), (4, 9, True),
                                          (0, 64, True), (0, 65, False)])
def test_small_layers_of_few_tokens_have_their_own(bits, B, taken, monkeypatch):
    layer, calls = fused_layer(bits), []
    finish = ops.expert_finish
    monkeypatch.setattr(ops, "expert_finish", lambda *a: calls.append(1) or finish(*a))
    layer.mlp.decode(torch.randn(B, 1, 512, device="cuda").bfloat16(), None,
                     layer.post_attention_layernorm,
                     torch.zeros(B, dtype=torch.int32, device="cuda"))
    assert bool(calls) == taken


@pytest.mark.parametrize("bits", [0, 4])
@pytest.mark.parametrize("B", [1, 8, 64, 65])
def test_layer(bits, B, monkeypatch):
    """A layer's step beside the one without them."""
    layer = fused_layer(bits)
    x = torch.randn(B, 1, 512, device="cuda").bfloat16()
    tickets = torch.zeros(B, dtype=torch.int32, device="cuda")
    norm, finish, calls = layer.post_attention_layernorm, ops.expert_finish, []
    monkeypatch.setattr(ops, "expert_begin_pays", lambda *a: True)
    monkeypatch.setattr(ops, "expert_finish", lambda *a: calls.append(1) or finish(*a))
    got = layer.mlp.decode(x, None, norm, tickets.clone()).double()
    assert bool(calls) == (B <= 64) and bool((tickets == 0).all())
    monkeypatch.setattr(ops, "expert_begin_ok", lambda *a: False)
    want = layer.mlp.decode(x, None, norm, tickets.clone()).double()
    # sums in other orders: a choice between experts that are nearly tied may differ
    off = (got - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)
    assert float(off.median()) < 0.01 and float((off > 0.01).float().mean()) < 0.1


def test_captured():
    """Replays of a captured step, with the step itself between them."""
    layer = fused_layer(4)
    x = torch.randn(20, 1, 512, device="cuda").bfloat16()
    norm = layer.post_attention_layernorm
    tickets = torch.zeros(20, dtype=torch.int32, device="cuda")

    def step():
        tickets.zero_()
        return layer.mlp.decode(x, None, norm, tickets)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, step())


def test_what_pays():
    """Ends of the rule, which looks at sizes alone."""
    w = lambda S: types.SimpleNamespace(shape=(0, S))  # noqa: E731
    for n, H, S, packed, pays in (
            (8, 2048, 64, True, True), (8, 2048, 2047, False, False), (8, 2048, 2048, False, True),
            (8, 2047, 64, True, False), (8, 1024, 4096, True, True), (8, 1024, 4095, True, False),
            (1, 128, 4097, False, True), (9, 128, 64, False, True)):
        assert ops.expert_begin_pays(n, H, None, w(S), packed) == pays
