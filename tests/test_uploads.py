"""Arrays of a batch on their way to the device."""

import numpy as np
import pytest
import torch

import tuvutar_cases as cases
from mlx_sharding_amd.ops.paged import RaggedBatch, PagedState, RowSpec, upload
from mlx_sharding_amd.parallel.batching import BatchEngine, Portion


@pytest.mark.parametrize("n", [0, 1, 7, 4096])
def test_upload_cpu(n):
    a = np.arange(n, dtype=np.int64)
    t = upload(a, "cpu")
    assert t.dtype == torch.int64 and t.tolist() == a.tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [0, 1, 1000])
def test_upload_behind_work(n):
    # many uploads while the stream is busy: none may find its memory taken
    x = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        x = x @ x / 64.0
    out = [upload(np.full(n, i, dtype=np.int32), "cuda") for i in range(200)]
    assert all(t.tolist() == [i] * n for i, t in enumerate(out))


@pytest.mark.gpu
@pytest.mark.parametrize("default", ["cpu", "meta", "cuda"])
def test_upload_with_a_default_device(default):
    with torch.device(default):
        t = upload(np.arange(5, dtype=np.int32), "cuda")
    assert t.device.type == "cuda" and t.tolist() == [0, 1, 2, 3, 4]


@pytest.mark.gpu
def test_batches_with_a_default_device():
    cfg = cases.config(32, 40, [cases.delta(2, 1, 16, 16, 4, ff=48)])
    model = cases.build(cfg, cases.weights(cfg), "cuda")
    steps = [[3, 1, 4, 1, 5], [9], [2]]
    want, got = BatchEngine(model, 128, 2), BatchEngine(model, 128, 2)
    for tokens in steps:
        portion = Portion("a", tokens, [len(tokens) - 1])
        a = want.step([portion])
        with torch.device("cuda"):
            b = got.step([portion])
        assert torch.equal(a, b)


class OnDevice:
    """A token as a scalar on a GPU shows itself to numpy."""

    def __init__(self, value):
        self.value = value

    def __array__(self, *args, **kwargs):
        raise TypeError("not on the host")

    def __int__(self):
        return self.value

    __index__ = __int__


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_tokens_that_are_scalars(device):
    cfg = cases.config(32, 40, [cases.delta(2, 1, 16, 16, 4, ff=48)])
    engine = BatchEngine(cases.build(cfg, cases.weights(cfg), device), 128, 2)
    scalar = OnDevice if device == "cpu" else lambda t: torch.tensor(t, device=device)
    tokens = [3, 1, 4]
    want = engine.step([Portion("a", tokens, [2])])
    got = engine.step([Portion("b", [scalar(t) for t in tokens], [2])])
    assert torch.equal(got, want)


def _places(device):
    state = PagedState([RowSpec(8)], 512, 3, torch.float32, torch.device(device))
    for r, n in enumerate((5, 64, 130)):
        state.admit(r)
        state.reserve(r, n + 3)
        state.live[r].length = n
    batch = RaggedBatch([(state.live[r], 1) for r in range(3)], device, wait=False)
    batch.advance()
    batch.advance()
    return batch


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_advance(device):
    b = _places(device)
    assert b.pos0.tolist() == b.tok_pos.tolist() == [7, 66, 132]
    assert b.cu.tolist() == [0, 1, 2, 3] and b.tok_entry.tolist() == [0, 1, 2]
    assert len(set(b.slots.tolist())) == 3 and b.max_pos == 133
