"""Queries, keys and values of few tokens from one kernel, beside the product and the rotations
one by one."""

import pytest
import torch

from mlx_sharding_amd import ops
from test_attend_few import cache_of, inputs, one_by_one

pytestmark = pytest.mark.gpu


# tiles of one to four and more than a round of them, groups of 16, 32 and 64 rows and one more,
# parts of a chunk; every size of a head
@torch.no_grad()
@pytest.mark.parametrize("M", [(1, 2), (4, 4), (1, 17), (8, 4), (3, 11), (1, 64)])
@pytest.mark.parametrize("H,heads,kv,D", [
    (32, 1, 1, 32), (96, 62, 1, 64), (544, 60, 2, 128), (160, 92, 2, 128), (1024, 28, 4, 256),
    (64, 62, 1, 256), (64, 125, 125, 64)])
@pytest.mark.parametrize("bias", [False, True])
def test_same_as_one_by_one(M, H, heads, kv, D, bias):
    (B, T), at = M, 5
    a = inputs(B, T, H, heads, kv, D, bias)
    here, there = cache_of(B, kv, D, at), cache_of(B, kv, D, at)
    order = ("x", "w", "b", "norm", "cos", "sin")
    got = ops.attend_few(*(a[n] for n in order), here, a["wo"], a["bo"], a["res"], heads,
                         D ** -0.5, 0.0, 0)
    assert got is not None
    want = one_by_one(*(a[n] for n in order), there, a["wo"], a["bo"], a["res"], heads,
                      D ** -0.5, 0.0, 0)
    # 32-bit sums in other orders may round the other way: one bf16 step, a turn two of them,
    # beside the dimension's partner
    for one, two in ((here.k, there.k), (here.v, there.v)):
        assert one.shape == two.shape
        size = torch.maximum(two.float().abs(), two.float().roll(D // 2, -1).abs())
        assert bool(((one.float() - two.float()).abs() <= size * 2.0 ** -6 + 1e-6).all())
        assert float((one != two).float().mean()) < 0.01
    assert here.offset == there.offset == at + T
    assert float((got.double() - want.double()).norm() / want.double().norm()) < 2.0 ** -9
