"""Latent attention of short portions over the cached rows themselves."""

from types import SimpleNamespace

import pytest
import torch

from mlx_sharding_amd.ops import ragged
from mlx_sharding_amd.ops.paged import PagedState, RaggedBatch, RowSpec

pytestmark = pytest.mark.gpu


# one key, a tile of 32 keys and a page of 64 less one, whole and more; slices of
# several tiles; tiles of 16 rows with remainders; rotated parts of one piece a
# thread, less and more; what lies behind a request's keys is not a number
@pytest.mark.parametrize("heads, rank, rot, dtype", [
    (16, 512, 64, torch.bfloat16), (3, 64, 32, torch.bfloat16),
    (5, 1024, 96, torch.bfloat16), (4, 128, 160, torch.float32),
])
def test_against_64_bits(heads, rank, rot, dtype):
    dev = torch.device("cuda")
    torch.manual_seed(heads)
    sh = ragged.LatentShape(heads, 32, rot, 32, rank)
    kept, new = (0, 30, 31, 32, 62, 63, 500, 2500), (1, 1, 2, 1, 1, 9, 16, 1)
    room = sum(-(-(a + b) // 64) * 64 for a, b in zip(kept, new))
    state = PagedState([RowSpec(sh.width)], room, len(kept), dtype, dev)
    rows = state.layers[0].rows
    rows.fill_(float("nan"))
    held = [state.admit(i) for i in range(len(kept))]
    for i, h in enumerate(held):
        state.reserve(i, kept[i] + new[i])
        h.length = kept[i]
        for j in range(kept[i] + new[i]):
            rows[h.pages[j // 64] * 64 + j % 64] = torch.randn(sh.width, device=dev)
    batch = [(h, n) for h, n in zip(held, new)]
    q = torch.randn(sum(new), heads * sh.dq, device=dev).to(dtype)
    q_abs = torch.randn(heads, sum(new), sh.rankp, device=dev).to(dtype)
    scale = sh.width ** -0.5
    got = ragged.latent_attention_absorbed(
        q, q_abs, state.layers[0], sh, scale, RaggedBatch(batch, dev), len(new),
        max(new)).cpu().double()
    want = ragged.latent_attention_absorbed(
        q.cpu().float(), q_abs.cpu().float(),
        SimpleNamespace(rows=rows.cpu().float()), sh, scale,
        RaggedBatch(batch, torch.device("cpu")), len(new), max(new)).double()
    # bf16: the result's own rounding, and that of the weights' two parts; float:
    # sums of up to 2501 products of weights that add up to 1
    bound = 2.0 ** -8 * 1.05 if dtype == torch.bfloat16 else 2.0 ** -18
    assert (got - want).abs().max() <= bound * want.abs().max()
