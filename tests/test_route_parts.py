"""A token's router in blocks of 16 experts, beside the one of one block, and the numbers
that a product clears for it."""

import types

import pytest
import torch

from mlx_sharding_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,E,top,H", [(1, 64, 6, 2048), (1, 1, 1, 128), (3, 17, 2, 8192),
                                       (64, 64, 6, 2048), (128, 48, 8, 2176),
                                       (5, 33, 33, 4096)])
@pytest.mark.parametrize("added", [False, True])
def test_same_as_one_block(N, E, top, H, added):
    g = torch.Generator("cuda").manual_seed(N + E)
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, res = randn(N, H).bfloat16(), randn(N, H).bfloat16() if added else None
    norm = types.SimpleNamespace(weight=(1 + 0.1 * randn(H)).bfloat16(), eps=1e-6,
                                 weight_offset=0.5)
    router = (randn(E, H) * 0.05).bfloat16()
    for scaling, normalize in ((1.5, True), (1.0, False)):
        one = ops.expert_route(x, res, norm, router, top, scaling, normalize)
        tickets = torch.zeros(N, dtype=torch.int32, device="cuda")
        parts = ops.expert_route(x, res, norm, router, top, scaling, normalize, tickets)
        assert torch.equal(one[1], parts[1])
        # the sum of squares has another order: one bf16 step of a normed value, which
        # may change the order of two experts that are nearly tied
        assert torch.allclose(one[0].float(), parts[0].float(), rtol=2.0 ** -7, atol=1e-6)
        p = torch.softmax(parts[0].double() @ router.double().T, -1)
        own = p.gather(1, parts[2].long())
        assert bool((parts[2].sort(-1).values.diff(dim=-1) > 0).all())
        assert bool(((own - p.topk(top, -1).values).abs() <= 1e-5).all())
        share = own / own.sum(-1, keepdim=True) if normalize else own
        assert bool(((parts[3].double() - scaling * share).abs() <= 1e-5).all())


def test_refused_numbers():
    x = torch.zeros(2, 128, dtype=torch.bfloat16, device="cuda")
    norm = types.SimpleNamespace(weight=x[0].clone(), eps=1e-6, weight_offset=0.0)
    for n, dtype in ((1, torch.int32), (2, torch.int64)):
        with pytest.raises(RuntimeError):
            ops.expert_route(x, None, norm, x.clone(), 1, 1.0, False,
                             torch.zeros(n, dtype=dtype, device="cuda"))


@pytest.mark.parametrize("M", [1, 12, 17, 64, 65])   # each kernel, and the library
@pytest.mark.parametrize("n", [1, 700])
def test_cleared(M, n):
    x = torch.randn(M, 2048, device="cuda").bfloat16()
    w = torch.randn(512, 2048, device="cuda").bfloat16()
    res = torch.randn(M, 512, device="cuda").bfloat16()
    numbers = torch.full((n + 2,), 7, dtype=torch.int32, device="cuda")
    y = ops.project(x, w, residual=res, clear=numbers[1:-1])
    assert numbers.tolist() == [7] + [0] * n + [7]
    assert torch.equal(y, ops.project(x, w, residual=res))
