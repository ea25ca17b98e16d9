"""Sums and maxima over the 64 lanes of a wave: each lane's value counts, once."""

import types

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [512, 2048])
def test_sums(H):
    """A norm's sum of squares from one column alone, for each of them."""
    x = torch.eye(H, device="cuda").bfloat16() * 3
    w = torch.ones(H, device="cuda").bfloat16()
    y = ops.rms_norm(x, w, 1e-6).double()
    expect = torch.eye(H, device="cuda").double() * H ** 0.5
    assert bool(((y - expect).abs() <= 2.0 ** -8 * expect).all())
    # and from all columns: twice a lane's value, or none, would show
    y = ops.rms_norm(torch.ones_like(x), w, 1e-6).double()
    assert bool(((y - 1).abs() <= 2.0 ** -8).all())


def test_maxima_and_sums_of_one_wave():
    """A router's largest score and sum of powers, with the largest in each lane."""
    E, H = 64, 128
    norm = types.SimpleNamespace(weight=torch.ones(H, device="cuda").bfloat16(),
                                 eps=0.0, weight_offset=0.0)
    x = torch.eye(H, device="cuda").bfloat16()[:E]       # normed: sqrt(128) = 11.3
    router = torch.eye(E, H, device="cuda").bfloat16() * 8 - 16
    _, _, choice, weight = ops.expert_route(x, None, norm, router, 1, 1.0, False)
    assert choice[:, 0].tolist() == list(range(E))
    assert bool((weight > 0.999999).all())
    flat = torch.full((3, H), 0.5, device="cuda").bfloat16()
    _, _, _, weight = ops.expert_route(flat, None, norm, torch.zeros_like(router), E,
                                       1.0, False)
    assert bool(((weight.double() - 1 / E).abs() <= 2.0 ** -23).all())


@pytest.mark.parametrize("S", [64 * 64, 64 * 64 - 17])
def test_maxima_of_slices(S):
    """Partial results of up to 64 slices of the keys, with the largest score in
    each."""
    D = 128
    ext = ops.hip_ext()
    v = torch.randn(1, 1, S, D, device="cuda").bfloat16()
    for at in range(31, S, 64):
        k = torch.zeros(1, 1, S, D, device="cuda").bfloat16()
        k[:, :, at, 0] = 60.0
        q = torch.zeros(1, 4, 1, D, device="cuda").bfloat16()
        q[..., 0] = 1.0
        out = ext.attn_decode(q, k, v, 1.0, 0.0, 0, None)
        # the other keys' weights are e^-60
        assert torch.equal(out[0, :, 0], v[0, :, at].expand(4, D)), at
