"""Latent attention of long portions on the prompt kernel, beside the general one."""

import pytest
import torch

from mlx_sharding_amd.ops import ragged
from mlx_sharding_amd.ops.paged import PagedState, RaggedBatch, RowSpec

pytestmark = pytest.mark.gpu


# short portions in front, tiles of 128 queries and 64 keys with remainders, one query
# more and less than a tile, continued requests; heads by eights or not
@pytest.mark.parametrize("heads", [8, 3])
def test_same_as_the_general_kernel(heads, monkeypatch):
    dev = torch.device("cuda")
    torch.manual_seed(heads)
    sh = ragged.LatentShape(heads, 128, 64, 128, 256)
    lens, more = (17, 128, 129, 1, 300, 64), (130, 20, 127, 5, 65, 2)
    room = sum(-(-(a + b) // 64) * 64 for a, b in zip(lens, more))
    state = PagedState([RowSpec(sh.width)], room, len(lens), torch.bfloat16, dev)
    state.layers[0].rows.normal_()
    held = [state.admit(i) for i in range(len(lens))]
    w_uk = (torch.randn(heads * sh.dimp, sh.rankp, device=dev) * 0.06).bfloat16()
    w_uv = (torch.randn(heads * sh.vdp, sh.rankp, device=dev) * 0.06).bfloat16()
    for i, h in enumerate(held):
        state.reserve(i, lens[i] + more[i])
    for part in (lens, more):
        order = sorted(range(len(part)), key=lambda i: part[i] > 16)
        b = RaggedBatch([(held[i], part[i]) for i in order], dev)
        q = torch.randn(sum(part), heads * sh.dq + 8, device=dev).bfloat16()[:, :heads * sh.dq]
        args = (q, state.layers[0], w_uk, w_uv, sh, 0.05, b)
        assert ragged._prompt_ext(q, sh) is not None
        got = ragged.latent_attention_expanded(*args).double()
        with monkeypatch.context() as m:
            m.setattr(ragged, "_prompt_ext", lambda *a: None)
            want = ragged.latent_attention_expanded(*args).double()
        # both round outputs to bf16, keys and values are the same
        size = want.abs().max()
        assert (got - want).abs().max() <= 2.0 ** -7 * size
        for i, h in enumerate(held):
            h.length += part[i]
