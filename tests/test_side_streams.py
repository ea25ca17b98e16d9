"""Layers on a stream of their own: inputs that it has yet to write, memory that other
streams use meanwhile."""

import pytest
import torch

from mlx_sharding_amd import ops
from test_module_calls import KINDS, a_layer

pytestmark = pytest.mark.gpu


def run(kind, fused):
    layer, cache, rope = a_layer(kind, fused)
    out = []
    for T in (140, 9, 1, 1):
        torch.manual_seed(T)
        big = torch.randn(2048, 2048, device="cuda")
        x = torch.randn(1, T, 256, device="cuda").bfloat16()
        angle = torch.rand(T, rope // 2, device="cuda")
        for _ in range(4):  # the input comes late
            big = big @ big * 1e-3
        x += (big[0, 0] * 0).nan_to_num().bfloat16()
        out.append(layer(x, torch.cos(angle), torch.sin(angle), cache))
    return out


@torch.no_grad()
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("kind", KINDS)
def test_same_on_another_stream(kind, fused):
    expect = run(kind, fused)
    torch.cuda.synchronize()
    side, busy = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = run(kind, fused)
    with torch.cuda.stream(busy):  # takes and fills memory as it becomes free
        for n in range(64):
            torch.full((1 << (8 + n % 12),), float("nan"), device="cuda")
    side.synchronize()
    busy.synchronize()
    for y, z in zip(got, expect):
        assert torch.equal(y, z)


@torch.no_grad()
def test_experts_of_a_prompt_on_another_stream():
    new = lambda *s: (torch.randn(*s, device="cuda") * 0.1).bfloat16()  # noqa: E731
    x, gate, up, down = new(500, 256), new(8, 128, 256), new(8, 128, 256), new(8, 256, 128)
    w, idx = torch.rand(500, 8, device="cuda").softmax(-1).topk(2)
    assert ops._tiles_ok(x, gate, up, down)
    expect = ops.grouped_expert_mlp(x, gate, up, down, w, idx)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        late = torch.zeros_like(x)
        big = torch.randn(2048, 2048, device="cuda")
        for _ in range(8):
            big = big @ big * 1e-3
        late.copy_(x)
        got = ops.grouped_expert_mlp(late, gate, up, down, w, idx)
    side.synchronize()
    assert torch.equal(got, expect)
