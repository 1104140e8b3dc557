"""Compensated attention with q and out in sequence order, and the tile
summaries from pooled features, against the tile-order form: layouts with
query tiles of one to four filled waves, an odd and an even number of steps
over the dropped tiles, and a subset of the heads in another order."""

import pytest
import torch

from miowtion_amd import kernels
from tests import helpers

pytestmark = pytest.mark.gpu

LAYOUTS = [dict(grid=(4, 16, 16), shape='2x8x8', text=0, extra=0),
           dict(grid=(3, 9, 11), shape='2x8x8', text=5, extra=3),
           dict(grid=(9, 13, 21), shape='2x4x16', text=200, extra=1)]


@pytest.mark.parametrize('kind', range(len(LAYOUTS)))
@pytest.mark.parametrize('heads', [None, [3, 0]])
def test_sequence_order_is_tile_order(kind, heads):
    spec = helpers.small_layout(**LAYOUTS[kind])
    lay, seq_len = helpers.product_layout(*spec, device='cuda'), spec[2]
    q, k, v = (t.cuda() for t in helpers.qkv(seq_len, 4, 128, seed=kind))
    heads = None if heads is None else torch.tensor(heads, device='cuda')
    hp, n = 4 if heads is None else heads.numel(), lay.n_tiles
    g = torch.Generator().manual_seed(kind)
    mask = (torch.rand(hp, n, n, generator=g) < 0.4).cuda()
    mask[:, torch.arange(n), torch.arange(n)] = True
    mask &= lay.kv_ok

    qt = kernels.gather_tiles(q, lay, heads)
    kt, feats_k = kernels.gather_and_pool(k, lay, heads)
    vt, feats_v = kernels.gather_and_pool(v, lay, heads)
    kc, vc = kernels.ops.summaries_from_means(feats_k, feats_v, lay.valid_count)
    want_kc, want_vc = kernels.tile_summaries(kt, vt, lay)
    # sums of at most 128 terms in another order, then one rounding to bf16:
    # next to a rounding boundary the two differ by one unit in the last place
    size = max(want_kc.abs().max().item(), 1e-6), max(want_vc.abs().max().item(), 1e-6)
    for got, want, top in ((kc, want_kc, size[0]), (vc, want_vc, size[1])):
        torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -14 * top)

    # the same summaries on both sides, then the same arithmetic: bit for bit
    lists = kernels.index_lists(mask, lay)
    tiles = kernels.ops.compensated_attention(qt, kt, vt, *lists, kc, vc, mask, lay.valid_count)
    want = torch.full((seq_len + 1, 4, 128), 7., dtype=torch.bfloat16, device='cuda')
    got = want.clone()
    kernels.scatter_tiles_(want, tiles, lay, heads)
    kernels.compensated_attention_seq_(got, q, kt, vt, feats_k, feats_v, mask, lists, lay, heads)
    assert torch.equal(got[:seq_len], want[:seq_len])
