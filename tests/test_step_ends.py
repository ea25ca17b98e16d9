"""What a captured decoding step begins and ends with."""

import pytest
import torch

from mlx_sharding_amd import ops
from mlx_sharding_amd.models.base import Linear, RMSNorm, head

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,W,half,scaled", [
    (1, 8, 1, False), (1, 64, 300, True),     # more rotations than vectors of a row
    (3, 2056, 32, True), (64, 4096, 64, False), (7, 3584, 128, True)])
def test_step_begin(rows, W, half, scaled):
    g = torch.Generator("cuda").manual_seed(rows)
    new = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    table, cos, sin = new(50, W).bfloat16(), new(9, half), new(9, half)
    scale = torch.tensor(W ** 0.5, dtype=torch.bfloat16, device="cuda") if scaled else None
    tokens = torch.randint(0, 50, (rows, 1), generator=g, device="cuda")
    tokens[0], tokens[-1] = 0, 49
    for p in (0, 8):
        pos = torch.tensor([p], dtype=torch.int32, device="cuda")
        h, c, s = ops.step_begin(tokens, table, scale, pos, cos, sin)
        want = torch.nn.functional.embedding(tokens, table)
        assert torch.equal(h, want if scale is None else want * scale)
        assert torch.equal(c, cos[p:p + 1]) and torch.equal(s, sin[p:p + 1])
    # outside of the tables
    tokens[0], pos[0] = 50, 9
    h, c, s = ops.step_begin(tokens, table, scale, pos, cos, sin)
    assert bool(h[0].isnan().all() and c.isnan().all() and s.isnan().all())
    assert not bool(h[1:].isnan().any())


def test_step_begin_leaves_other_forms():
    t = torch.zeros(2, 1, dtype=torch.int64, device="cuda")
    pos = torch.zeros(1, dtype=torch.int32, device="cuda")
    rot = torch.zeros(4, 8, device="cuda")
    table = torch.zeros(5, 16, dtype=torch.bfloat16, device="cuda")
    for args in ((t.int(), table), (t, table.float()), (t, table[:, :8]),
                 (t.expand(2, 2), table), (t, table[:, 1:13].contiguous())):
        assert ops.step_begin(*args, None, pos, rot, rot) is None


@pytest.mark.parametrize("rows,n", [(1, 1), (2, 1023), (64, 1025), (5, 32000)])
def test_step_end(rows, n):
    x = torch.randn(rows, 2, n, device="cuda").bfloat16()
    pos = torch.tensor([41], dtype=torch.int32, device="cuda")
    y = ops.step_end(x[:, -1, :], pos)
    assert y.dtype == torch.float32 and torch.equal(y, x[:, -1].float())
    assert int(pos) == 42


# normed rows and results rounded to bf16: below 4e-3 of the result's 2-norm
@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65])
@pytest.mark.parametrize("V", [1000, 32768, 32784])   # up to 2^26 weights, and more
def test_head(rows, V, monkeypatch):
    K, fused = 2048, []
    g = torch.Generator("cuda").manual_seed(V)
    new = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    norm, out = RMSNorm(K, 1e-5, 1.0).cuda(), Linear(K, V).cuda()
    norm.weight.data = (new(K) * 0.1).bfloat16()
    out.weight.data = (new(V, K) * K ** -0.5).bfloat16()
    x = new(rows, 1, K).bfloat16()
    h = x.double()
    h = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5)
    want = (h * (norm.weight.double() + 1)) @ out.weight.double().t()
    project = ops.project
    monkeypatch.setattr(ops, "project", lambda *a, **k: (fused.append(k["norm"]),
                                                         project(*a, **k))[1])
    for got in (head(norm, x, out), head(norm, x, table=out.weight)):
        assert got.shape == (rows, 1, V)
        assert float((got.double() - want).norm() / want.norm()) < 4e-3
    # the norm goes with the product, or before the library's
    assert fused == [norm] * (2 if rows <= 32 or (rows <= 64 and V <= 32768) else 0)
