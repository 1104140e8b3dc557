"""The top-k's order among equal scores that lie in different lanes of its
wave, against the oracle."""

import types

import pytest
import torch

from miowtion_amd import mask as pm
from oracle import mask as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [64, 65, 200, 1100])
def test_topk_ties_across_lanes(n):
    """Few distinct scores, so that most rounds of the top-k find the same
    score in several lanes."""
    g = torch.Generator().manual_seed(n)
    scores = torch.randint(0, 3, (2, n, n), generator=g).float() - 1
    scores[0, :, ::7] = float('-inf')
    scores[1, ::2, ::5] = float('nan')
    scores[1, 1::2, ::3] = float('inf')
    kv_ok = torch.ones(n, dtype=torch.bool)
    lay = types.SimpleNamespace(n_video_tiles=n, kv_ok=kv_ok)
    block = om.ColumnBlock(0, n, om.Budget(ratio=0.4), n * 128)
    ri, rk = om.select_video_blocks(scores, lay, [block])
    glay = types.SimpleNamespace(n_video_tiles=n, kv_ok=kv_ok.cuda())
    gblock = pm.ColumnBlock(0, n, pm.Budget(ratio=0.4), n * 128)
    for rows in (None, torch.arange(n, device='cuda')):
        sel = pm.select_video_blocks(scores.cuda(), glay, [gblock], rows)
        assert torch.equal(sel.index.cpu(), ri) and torch.equal(sel.keep.cpu(), rk)
