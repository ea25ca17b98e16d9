"""Experts of a prompt's tokens, and what is added to their sum, in one kernel each."""

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,E,top", [(1, 1, 1), (5, 64, 64), (131, 7, 3), (1030, 64, 6),
                                     (4, 64, 1)])
@pytest.mark.parametrize("normalize", [False, True])
def test_choice(N, E, top, normalize):
    g = torch.Generator("cuda").manual_seed(N)
    logits = torch.randn(N, E, generator=g, device="cuda")
    # no two equal: choices are then unique
    logits = (logits.argsort(-1).argsort(-1).float() / 8).bfloat16()
    w, idx = ops.moe_gate(logits, top, routed_scaling_factor=1.5, norm_topk_prob=normalize)
    want, want_idx = ref.moe_gate(logits.double(), top, routed_scaling_factor=1.5,
                                  norm_topk_prob=normalize)
    assert w.dtype == torch.float32 and torch.equal(idx, want_idx)
    # exponential, sum and quotients in 24 bits
    assert torch.allclose(w, want.float(), rtol=2e-5, atol=1e-9)


def test_choice_of_ties_and_no_numbers():
    logits = torch.zeros(3, 9, dtype=torch.bfloat16, device="cuda")
    logits[1], logits[2, 4] = float("-inf"), float("nan")
    _, idx = ops.moe_gate(logits, 3)
    assert idx.tolist() == [[0, 1, 2]] * 3     # in their order, each once


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_weights_keep_their_bits(spread, normalize):
    g = torch.Generator("cuda").manual_seed(1)
    logits = (torch.randn(4096, 64, generator=g, device="cuda") * spread).bfloat16()
    w = ops.moe_gate(logits, 6, norm_topk_prob=normalize)[0].double()
    want = torch.softmax(logits.double(), -1).topk(6, -1).values
    if normalize:
        want = want / want.sum(-1, keepdim=True)
    # in units of 2^-24, each a rounding: the exponential two, its sum over 64 lanes six,
    # the quotient two; the second sum and quotient as many less the exponential
    off = (w.sort(-1, descending=True).values - want).abs() / want
    assert float(off.max()) < (18 if normalize else 10) * 2 ** -24


def test_no_choice():
    w, idx = ops.moe_gate(torch.zeros(3, 9, dtype=torch.bfloat16, device="cuda"), 0)
    assert w.shape == idx.shape == (3, 0) and idx.dtype == torch.int64


@pytest.mark.parametrize("top", [1, 2, 3, 4, 6, 7, 9])
@pytest.mark.parametrize("H", [4, 1028, 2048])
def test_sum(top, H):
    N = 70
    g = torch.Generator("cuda").manual_seed(top)
    new = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    d, w = new(N * top, H).bfloat16(), new(N, top)
    pos = torch.randperm(N * top, generator=g, device="cuda").view(N, top).int()
    more = [new(N, H).bfloat16() for _ in range(2)]
    for n in range(3):
        want = (d.double()[pos.long()] * w.double()[..., None]).sum(1)
        want = sum((t.double() for t in more[:n]), want)
        got = ops.hip_ext().moe_gather_reduce(d, pos, w, N, *more[:n])
        # one rounding to 8 bits, and 2^-24 of the terms for each sum
        assert bool(((got.double() - want).abs() <= want.abs() * 2 ** -8 + 1e-4).all())


@pytest.mark.parametrize("form", ["rows", "strided", "float", "three"])
def test_rows_beside_the_experts(form):
    N, E, H, I = 300, 4, 128, 128
    g = torch.Generator("cuda").manual_seed(1)
    new = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    x, stacks = new(N, H), [new(E, I, H) * 0.1, new(E, I, H) * 0.1, new(E, H, I) * 0.1]
    w = torch.rand(N, 2, generator=g, device="cuda")
    idx = torch.rand(N, E, generator=g, device="cuda").topk(2).indices
    plus = [new(N, H), new(N, H)]
    if form == "strided":
        plus[1] = new(N, 2 * H)[:, :H]
    elif form == "float":
        plus[0] = plus[0].float()
    elif form == "three":
        plus.append(new(N, H))
    alone = ops.grouped_expert_mlp(x, *stacks, w, idx)
    got = ops.grouped_expert_mlp(x, *stacks, w, idx, plus)
    want = alone
    for t in plus:
        want = want + t
    assert got.dtype == want.dtype
    # roundings of the sums in between
    assert torch.allclose(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -6)
