"""Queries, keys and values of new tokens in one kernel, beside the separate ones."""

import math

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.ops.kvcache import KVCache

pytestmark = pytest.mark.gpu
EXT = ops.hip_ext()


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("B,T,Hq,Hkv,D", [(1, 1, 1, 1, 16), (3, 1, 8, 2, 64), (64, 1, 32, 8, 128),
                                          (1, 57, 32, 4, 64), (2, 300, 4, 2, 256),
                                          (1, 9, 3, 1, 24)])  # the last: apart
def test_same_as_separate_kernels(B, T, Hq, Hkv, D, captured, monkeypatch):
    torch.manual_seed(D + T)
    rows = torch.randn(B, T, (Hq + 2 * Hkv) * D, device="cuda").bfloat16()
    q, k, v = (t.view(B, T, -1, D) for t in rows.split([Hq * D, Hkv * D, Hkv * D], -1))
    angle = torch.rand(T, D // 2, device="cuda") * 2 * math.pi
    cos, sin = torch.cos(angle), torch.sin(angle)
    caches = []
    for _ in range(2):
        c = KVCache(Hkv, D, D, torch.bfloat16, torch.device("cuda"))
        c._ensure(B, T + 20)
        c._k.fill_(math.nan)
        c._v.fill_(math.nan)
        c.offset = 7
        if captured:
            c.graph_pos = torch.tensor([7], dtype=torch.int32, device="cuda")
        caches.append(c)
    one, two = caches
    ran = []

    class Spied:
        def __getattr__(self, name):
            ran.append(name)
            return getattr(EXT, name)

    with monkeypatch.context() as m:
        m.setattr(ops, "hip_ext", Spied)
        got = one.append_rope_qkv(q, k, v, cos, sin)
    assert ran == (["rope_qkv"] if D % 16 == 0 else ["rope_append_kv"])
    want = (ops.apply_rope(q, cos, sin), *two.append_rope_kv(k, v, cos, sin))
    for a, b in zip((*got, one._k, one._v), (*want, two._k, two._v)):
        # a turn's two products may be contracted the other way round: one bf16 step
        assert a.shape == b.shape and torch.allclose(
            a.float(), b.float(), rtol=2.0 ** -7, atol=1e-6, equal_nan=True)
    assert torch.equal(one._v.view(torch.int16), two._v.view(torch.int16))
    assert one.offset == two.offset
