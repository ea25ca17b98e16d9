"""Choice and placement of few tokens' experts in one kernel, beside the two kernels."""

import pytest
import torch

from mlx_sharding_amd.ops.ragged import hip_ragged

pytestmark = pytest.mark.gpu


# one block of tokens and more, experts of every lane and more, experts that are identities,
# tiles of one pair, some and all
@pytest.mark.parametrize("N", [1, 5, 15, 16, 17, 70])
@pytest.mark.parametrize("total,experts,top", [(64, 64, 6), (64, 50, 8), (1, 1, 1), (17, 16, 17),
                                               (65, 65, 4)])
@pytest.mark.parametrize("tile", [1, 16, 128])
@pytest.mark.parametrize("on_input", [False, True])
def test_same_as_two_kernels(N, total, experts, top, tile, on_input):
    g = torch.Generator("cuda").manual_seed(N + total)
    K, ext = 256, hip_ragged()
    h = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    w = torch.randn((total + 15) // 16, K // 32, 64, 8, generator=g, device="cuda").bfloat16()
    args = (h, w, None, total, experts, top, False, True)
    idx, weight, rank, hist = ext.expert_route(*args)
    _, _, tiles, used, _ = ext.expert_plan(idx, rank, hist, None, experts, tile)
    got_w, where, tokens, got_tiles, got_used, scale = ext.expert_place(*args, on_input, tile)
    assert torch.equal(got_w, weight)
    assert torch.equal(got_tiles, tiles) and torch.equal(got_used, used)
    # the order of an expert's pairs is any
    placed = idx < experts
    assert torch.equal(where >= 0, placed)
    at = where[placed].long()
    assert torch.equal(at.sort().values, torch.arange(len(at), device="cuda"))
    assert torch.equal(tokens[at], torch.arange(N, device="cuda").int()[:, None]
                       .expand(N, top)[placed])
    assert torch.equal(idx[placed][at.argsort()], idx[placed].sort().values)
    assert (scale is None) != on_input
    if on_input:
        assert torch.equal(scale[at], weight[placed])
