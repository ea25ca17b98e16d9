"""What a 32-bit residual stream begins with, and steps that want all rows."""

import pytest
import torch
import torch.nn.functional as F

import dufinex_cases as cases
from mlx_sharding_amd.ops.ragged import token_rows
from mlx_sharding_amd.parallel.batching import BatchEngine, Portion


@pytest.mark.gpu
@pytest.mark.parametrize("N,W", [(1, 8), (3, 2048), (300, 264)])
def test_rows(N, W):
    g = torch.Generator("cuda").manual_seed(N)
    table = torch.randn(40, W, generator=g, device="cuda").bfloat16()
    tokens = torch.randint(0, 40, (N,), generator=g, device="cuda")
    tokens[0], tokens[-1] = 39, 0
    assert torch.equal(token_rows(tokens, table), F.embedding(tokens, table).float())
    assert torch.equal(token_rows(tokens, table, 50.0),
                       F.embedding(tokens, table).float() * 50.0)
    tokens[0] = 40
    got = token_rows(tokens, table)
    assert bool(got[0].isnan().all()) and not bool(got[1:].isnan().any())


@pytest.mark.gpu
def test_other_forms():
    table = torch.randn(9, 32, device="cuda").bfloat16()
    t = torch.tensor([[1, 8], [0, 3]], device="cuda")
    for tokens, rows in ((t, table), (t.int(), table), (t.t(), table), (t, table.float()),
                         (t, table[:, :12]), (t, table[:, 1:25].contiguous()),
                         (t[:, :0], table)):
        assert torch.equal(token_rows(tokens, rows, 2.0),
                           F.embedding(tokens, rows).float() * 2.0)


def test_cpu():
    table, t = torch.randn(5, 7), torch.tensor([4, 0])
    assert torch.equal(token_rows(t, table, 3.0), F.embedding(t, table) * 3.0)


def test_all_rows_wanted(monkeypatch):
    """Rows are selected only where some of them, or another order, are wanted."""
    cfg = next(iter(cases.CONFIGS.values()))
    m = cases.build(cfg, cases.weights(cfg), "cpu", torch.float32)
    engine, alone = BatchEngine(m, 256, 4), BatchEngine(m, 256, 4)
    asked, run = [], m.run

    def seen(x, batch, state, rows=None):
        asked.append(rows if rows is None else rows.tolist())
        return run(x, batch, state, rows=rows)

    monkeypatch.setattr(m, "run", seen)
    steps = [[Portion("a", [5], [0]), Portion("b", [6], [0])], [Portion("a", [7, 8], [0, 1])],
             [Portion("b", [9, 3], [1])], [Portion("b", [1, 2], [1, 0])],
             [Portion("a", [4], []), Portion("b", [4], [0])]]
    got = [engine.step(s) for s in steps]
    assert asked == [None, None, [1], [1, 0], [1]]
    for s, g in zip(steps, got):  # each place of a portion by itself
        want = []
        for p in s:
            z = [alone.step([Portion(p.rid, [t], [0])])[0] for t in p.tokens]
            want += [z[w] for w in p.want]
        torch.testing.assert_close(g, torch.stack(want), atol=1e-4, rtol=1e-4)
