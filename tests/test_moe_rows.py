"""Routed experts of a decoding step, against 64 bits."""

import types

import pytest
import torch
import torch.nn.functional as F

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


def stack(E, O, K, bits, gs, gen):
    """(matrices as ops.expert_rows takes them, their values in 64 bits)"""
    if bits == 16:
        w = (torch.randn(E, O, K, generator=gen, device="cuda") * 0.03).bfloat16()
        return [w], w.double()
    words = torch.randint(0, 2 ** 32, (E, O, K * bits // 32), generator=gen,
                          device="cuda").to(torch.uint32)
    new = lambda std: (torch.randn(E, O, K // gs, generator=gen,  # noqa: E731
                                   device="cuda") * std).bfloat16()
    s, b = new(0.0025 if bits == 4 else 0.00016), new(0.005)
    shifts = torch.arange(0, 32, bits, device="cuda")
    q = (words.view(torch.int32).to(torch.int64)[..., None] >> shifts) & (2 ** bits - 1)
    q = q.reshape(E, O, K // gs, gs).double()
    return [words, s, b], (q * s.double()[..., None] + b.double()[..., None]).flatten(-2)


@pytest.mark.parametrize("N,E,top,I,H,bits,gs", [
    (1, 8, 2, 128, 256, 4, 64),        # fewer units than waves, pairs than experts
    (3, 5, 5, 384, 1152, 16, 128),     # all experts, nine units
    (33, 3, 2, 128, 128, 4, 128),      # one unit; groups of 16 tokens and a rest
    (128, 64, 6, 256, 512, 8, 32),     # most tokens
    (100, 4, 1, 256, 384, 4, 32), (16, 64, 8, 1408, 2048, 8, 64),
    (64, 64, 6, 1408, 2048, 4, 64), (17, 16, 4, 1536, 5120, 4, 128),
    (9, 16, 4, 1536, 3072, 16, 128), (128, 1, 1, 128, 640, 8, 128)])
def test_experts(N, E, top, I, H, bits, gs):
    gen = torch.Generator("cuda").manual_seed(N + H)
    randn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    gate, gd = stack(E, I, H, bits, gs, gen)
    up, ud = stack(E, I, H, bits, gs, gen)
    down, dd = stack(E, H, I, bits, gs, gen)
    x, res, shared = (randn(N, H).bfloat16() for _ in range(3))
    norm = types.SimpleNamespace(weight=(1 + 0.1 * randn(H)).bfloat16(), eps=1e-6,
                                 weight_offset=0.5)
    router = (randn(E, H) * 0.05).bfloat16()
    assert ops.expert_rows_ok(x, router, up[0], down[0], top, bits, gs)
    y, h, choice, weight = ops.expert_route(x, res, norm, router, top, 1.5, True)
    hd = (x.double() + res.double()).bfloat16()
    assert torch.equal(h, hd)
    yd = hd.double()
    yd = yd * torch.rsqrt(yd.pow(2).mean(-1, keepdim=True) + 1e-6)
    yd = yd * (norm.weight.double() + 0.5)
    assert bool(((y.double() - yd).abs() <= 2.0 ** -8 * yd.abs() + 1e-6).all())

    # chosen experts are the largest, up to 32-bit sums over H products
    p = torch.softmax(y.double() @ router.double().T, -1)
    own, best = p.gather(1, choice.long()), p.topk(top, -1).values
    assert bool((choice.sort(-1).values.diff(dim=-1) > 0).all())
    assert bool(((own - best).abs() <= 1e-5).all())
    share = 1.5 * own / own.sum(-1, keepdim=True)
    assert bool(((weight.double() - share).abs() <= 1e-5).all())

    rows = ops.expert_rows(y, choice, weight, gate, up, down, bits, gs).double()
    e, a = choice.long().flatten(), y.double().repeat_interleave(top, 0)
    # weights and units are rounded to fp16 (2^-11 each) or units to bf16 (2^-8)
    wide = bits == 16
    uw, uh = (0.0, 2.0 ** -8) if wide else (2.0 ** -11, 2.0 ** -11)
    tiny = H * 2.0 ** -24
    for i in range(0, N * top, 64):
        j = slice(i, i + 64)
        dot = lambda m, v: torch.bmm(m[e[j]], v[..., None])[..., 0]  # noqa: E731
        g, u = dot(gd, a[j]), dot(ud, a[j])
        size = lambda m: dot(m.abs(), a[j].abs()) * (2 * uw + tiny)  # noqa: E731
        unit = F.silu(g) * u
        off = 1.1 * size(gd) * (u.abs() + size(ud)) + F.silu(g).abs() * size(ud)
        off = off + uh * unit.abs() + 6e-8
        w = weight.double().flatten()[j, None]
        expect = w * dot(dd, unit)
        bound = w * (dot(dd.abs(), off) + dot(dd.abs(), unit.abs()) * (2 * uw + tiny))
        assert bool(((rows[j] - expect).abs() <= bound + 1e-6).all())

    out = ops.expert_sum(rows.float(), h, shared, N).double()
    total = h.double() + shared.double() + rows.view(N, top, H).sum(1)
    assert bool(((out - total).abs() <= 2.0 ** -8 * total.abs() + 1e-5).all())
    alone, terms = ops.expert_sum(rows.float(), None, None, N).double(), rows.view(N, top, H)
    total = terms.sum(1)
    # rounded once to bf16, from 32-bit sums in any order
    bound = 2.0 ** -8 * total.abs() + top * 2.0 ** -24 * terms.abs().sum(1)
    assert bool(((alone - total).abs() <= bound).all())


# Units of 128 of the contraction, of which eight waves have as many or one less each: 25 to
# 40, one wave's last one missing, most waves' and none; in either product.  Up to 64 pairs
# and more.
@pytest.mark.parametrize("N,E,top", [(5, 3, 2), (70, 2, 1)])
@pytest.mark.parametrize("units,bits,gs", [
    (25, 4, 64), (28, 4, 32), (31, 4, 128), (25, 8, 128), (28, 8, 64), (31, 8, 32),
    (32, 4, 64), (33, 8, 64), (36, 4, 128), (39, 8, 32), (9, 4, 64), (15, 8, 64),
    (17, 4, 32), (20, 8, 128), (23, 4, 64), (15, 16, 128), (17, 16, 128), (20, 16, 128)])
def test_units_that_some_waves_lack(N, E, top, units, bits, gs):
    test_experts(N, E, top, 384, units * 128, bits, gs)
    test_experts(N, E, top, units * 128, 384, bits, gs)


def test_ties_and_rows_that_are_no_numbers():
    """Equal scores: the first experts.  NaN: some experts, each once."""
    H, E, top = 256, 12, 4
    norm = types.SimpleNamespace(weight=torch.ones(H, device="cuda").bfloat16(),
                                 eps=1e-6, weight_offset=0.0)
    x = torch.ones(3, H, device="cuda").bfloat16()
    x[1] = float("nan")
    router = torch.zeros(E, H, device="cuda").bfloat16()
    router[7] = 1.0
    _, _, choice, weight = ops.expert_route(x, None, norm, router, top, 1.0, False)
    assert choice[0].tolist() == [7, 0, 1, 2] == choice[2].tolist()
    assert choice[1].sort().values.tolist() == [0, 1, 2, 3]
    assert bool(weight[1].isnan().all())


def test_layer_as_before():
    """A decoder layer's step on these kernels beside the general path."""
    from mlx_sharding_amd.config import ModelConfig
    from mlx_sharding_amd.models.deepseek_v2 import DeepseekV2MoE
    for bits in (4, 8, 0):
        raw = {"model_type": "deepseek_v2", "hidden_size": 512,
               "moe_intermediate_size": 256, "n_routed_experts": 16,
               "num_experts_per_tok": 3, "n_shared_experts": 1,
               "intermediate_size": 256}
        if bits:
            raw["quantization"] = {"group_size": 64, "bits": bits}
        cfg = ModelConfig.from_dict(raw)
        q = cfg.quantization
        torch.manual_seed(bits)
        with torch.device("cuda"):
            moe = DeepseekV2MoE(cfg, lambda p: q, "m")
        for name, p in moe.named_parameters():
            if p.is_floating_point():
                std = {"scales": 0.0025 / 16 ** (bits == 8), "biases": 0.005}
                p.data.normal_(0, std.get(name.rsplit(".", 1)[-1], 0.05))
            else:
                p.data.random_(0, 2 ** 31 - 1)
            p.requires_grad_(False)
        norm = types.SimpleNamespace(weight=torch.ones(512, device="cuda").bfloat16(),
                                     eps=1e-6, weight_offset=0.0)
        for B, T in ((1, 1), (40, 1), (2, 9)):
            x = torch.randn(B, T, 512, device="cuda").bfloat16()
            assert moe.decodes(x)
            got = moe.decode(x, None, norm).double()
            # the same choice: where two experts are nearly tied, the general
            # path's bf16 scores may fall the other way
            y, _, choice, weight = ops.expert_route(
                x.view(-1, 512), None, norm, moe.gate.weight, 3, 1.0, False)
            rest = moe.switch_mlp(y, weight, choice.long()) + moe.shared_experts(y)
            expect = x.double() + rest.double().view_as(x)
            assert got.shape == x.shape
            assert (got - expect).norm() < 0.01 * expect.norm()


def decoder_layer(bits=0, I=256, seed=0):
    """A decoder layer with 16 routed experts and a shared one, of random weights."""
    from mlx_sharding_amd.config import ModelConfig
    from mlx_sharding_amd.models.deepseek_v2 import DeepseekV2DecoderLayer
    raw = {"model_type": "deepseek_v2", "hidden_size": 512,
           "moe_intermediate_size": I, "n_routed_experts": 16,
           "num_experts_per_tok": 3, "n_shared_experts": 1, "intermediate_size": 256,
           "num_attention_heads": 4, "kv_lora_rank": 64, "qk_nope_head_dim": 32,
           "qk_rope_head_dim": 16, "v_head_dim": 32, "first_k_dense_replace": 0}
    if bits:
        raw["quantization"] = {"group_size": 64, "bits": bits}
    cfg = ModelConfig.from_dict(raw)
    torch.manual_seed(seed)
    with torch.device("cuda"):
        layer = DeepseekV2DecoderLayer(
            cfg, lambda p: cfg.quantization if "switch" in p else None, "m", 0)
    for name, p in layer.named_parameters():
        kind = name.rsplit(".", 1)[-1]
        if not p.is_floating_point():
            p.data.random_(0, 2 ** 31 - 1)
        elif "layernorm" in name:
            p.data.normal_(1.0, 0.1)
        else:
            p.data.normal_(0, {"scales": 0.0025 / 16 ** (bits == 8),
                               "biases": 0.005}.get(kind, 0.05))
    return layer


def one_position(rope=16):
    angle = torch.rand(1, rope // 2, device="cuda")
    return torch.cos(angle), torch.sin(angle)


@pytest.mark.parametrize("B", [8, 100])
def test_layer_takes_slices(B):
    """Hidden states as the last token of longer ones, and off 16 bytes."""
    layer = decoder_layer()
    turn = one_position()
    big = torch.randn(B, 3, 512, device="cuda").bfloat16()
    x = big[:, -1:]
    assert layer.mlp.decodes(x)
    expect = layer(x.contiguous(), *turn, None)
    assert torch.equal(layer(x, *turn, None), expect)
    odd = torch.empty(B * 512 + 1, device="cuda").bfloat16()[1:].view(B, 1, 512)
    odd.copy_(x)
    assert torch.equal(layer(odd, *turn, None), expect)


@pytest.mark.parametrize("bits", [4, 8])
def test_experts_loaded_later(bits):
    """Words, scales and biases that are loaded behind the first step, written where
    they lie or put in place of the old ones, are what the next step takes."""
    layer, other = decoder_layer(bits, seed=1), decoder_layer(bits, seed=2)
    turn = one_position()
    x = torch.randn(8, 1, 512, device="cuda").bfloat16()
    assert layer.mlp.decodes(x)
    before = layer(x, *turn, None)
    theirs = dict(other.named_parameters())
    for name, p in layer.named_parameters():
        if "switch" not in name:
            theirs[name].data.copy_(p)
    for kind in ("scales", "biases", "weight"):
        for name, p in layer.named_parameters():
            if name.endswith("switch_mlp.down_proj." + kind):
                p.copy_(theirs[name])
            elif "switch" in name and name.endswith(kind):
                p.data = theirs[name].detach().clone()
        got = layer(x, *turn, None)
        fresh = decoder_layer(bits, seed=3)
        fresh.load_state_dict(layer.state_dict())
        assert torch.equal(got, fresh(x, *turn, None))
        assert not torch.equal(got, before)
        before = got
    assert torch.equal(got, other(x, *turn, None))


@pytest.mark.parametrize("bits,I", [(4, 192), (8, 64), (0, 320)])
def test_widths_of_the_general_kernels(bits, I):
    """Experts that are no multiple of 128 wide are chosen and sorted in one kernel and
    run by ranges of tokens."""
    layer = decoder_layer(bits, I)
    moe = layer.mlp
    for n in (1, 8, 100):
        x = torch.randn(n, 1, 512, device="cuda").bfloat16()
        assert not moe.decodes(x)
        got = moe(x).double().view(n, 512)
        flat = x.view(n, 512)
        logits = moe.gate(flat).double()
        weight, chosen = torch.softmax(logits, -1).topk(3, -1)
        e, a = chosen.flatten(), flat.double().repeat_interleave(3, 0)
        gate, up, down = (m.dense().double() for m in (
            moe.switch_mlp.gate_proj, moe.switch_mlp.up_proj, moe.switch_mlp.down_proj))
        dot = lambda m, v: torch.bmm(m[e], v[..., None])[..., 0]  # noqa: E731
        rows = dot(down, F.silu(dot(gate, a)) * dot(up, a)) * weight.flatten()[:, None]
        expect = rows.view(n, 3, 512).sum(1) + moe.shared_experts(flat).double()
        # units, rows and sums are rounded to bf16 or fp16
        assert (got - expect).norm() < 0.01 * expect.norm()
