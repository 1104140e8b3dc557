"""The block lists built in one kernel, bit for bit against the oracle and
against the kernels they stand for: the transposed (Q-direction) lists over
sizes around a 64-tile group and past one chunk of staged rows, and the lists
straight from a selection against the mask and its lists. Key tiles without a
real row, full and partial ones, empty and whole rows and columns."""

import types

import pytest
import torch

from miowtion_amd import kernels
from miowtion_amd import mask as pm
from miowtion_amd import ops
from oracle import mask as om
from tests import helpers

pytestmark = pytest.mark.gpu


def _tables(n, g):
    kv_ok = torch.rand(n, generator=g) < 0.9
    return kv_ok, kv_ok & (torch.rand(n, generator=g) < 0.6)


@pytest.mark.parametrize('rows,n,density', [(1, 1, 0.5), (63, 63, 0.1), (64, 64, 0.5), (65, 65, 0.9),
                                            (130, 130, 0.0), (130, 7, 1.0), (4096, 3, 0.3),
                                            (4097, 3, 0.3), (8300, 66, 0.02)])
def test_transposed_lists_match_oracle(rows, n, density):
    g = torch.Generator().manual_seed(rows + n)
    mask = torch.rand(2, rows, n, generator=g) < density
    if rows > 2:
        mask[0, 1] = True
        mask[1, :, 0] = True
    kv_ok, full = _tables(n, g)
    got = ops.index_lists_t(mask.cuda(), kv_ok.cuda(), full.cuda())
    want = om.index_lists(mask, types.SimpleNamespace(kv_ok=kv_ok, full_tile=full), transpose=True)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and torch.equal(a.cpu(), b)


@pytest.mark.parametrize('n,n_video,k', [(1, 1, 1), (64, 64, 9), (65, 40, 40), (200, 129, 5),
                                         (4096, 4000, 70)])
def test_selection_lists_match_the_mask_and_its_lists(n, n_video, k):
    g = torch.Generator().manual_seed(n + k)
    heads = 2 if n < 1000 else 1
    index = torch.rand(heads, n_video, n_video, generator=g).topk(k, -1)[1]
    keep = torch.rand(heads, n_video, k, generator=g) < 0.8
    kv_ok, full = (t.cuda() for t in _tables(n, g))
    index, keep = index.cuda(), keep.cuda()
    mask = ops.dense_block_mask(index, keep, kv_ok, n_video, True)
    for a, b in zip(ops.selection_lists(index, keep, kv_ok, full, n_video),
                    ops.index_lists(mask, kv_ok, full)):
        assert torch.equal(a, b)
    # a selection that is a column slice of a wider one
    for a, b in zip(ops.selection_lists(index[..., :1], keep[..., :1], kv_ok, full, n_video),
                    ops.index_lists(ops.dense_block_mask(index[..., :1], keep[..., :1], kv_ok, n_video,
                                                         True), kv_ok, full)):
        assert torch.equal(a, b)


def test_selection_lists_of_a_layout_and_refusals():
    spec = helpers.small_layout()
    lay = helpers.product_layout(*spec, device='cuda')
    scores = torch.rand(3, lay.n_video_tiles, lay.n_tiles, device='cuda')
    sel = pm.select_video_blocks(scores, lay, pm.column_blocks(lay, pm.Budget(ratio=0.3)))
    want = kernels.index_lists(pm.dense_block_mask(sel, lay), lay)
    for a, b in zip(kernels.selection_lists(sel, lay), want):
        assert torch.equal(a, b)
    with pytest.raises(ValueError, match='all video rows'):
        ops.selection_lists(sel.index[:, 1:], sel.keep[:, 1:], lay.kv_ok, lay.full_tile,
                            lay.n_video_tiles)
    with pytest.raises(NotImplementedError):
        ops.index_lists_t(torch.zeros(1, 2, 2, dtype=torch.bool), lay.kv_ok.cpu()[:2],
                          lay.full_tile.cpu()[:2])
