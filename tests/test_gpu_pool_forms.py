"""The pooled gather's two forms (one wave per tile and head group, or the
tile's slots split over waves) give the same bits: a launch of few heads or
tiles takes one form, a launch of many the other, and a layer's heads come in
any chunks. Heads that do not fill a group, partial tiles, both head_dims."""

import pytest
import torch

from miowtion_amd import kernels
from oracle import predictor as op
from oracle import tiling as ot
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dim', [64, 128])
@pytest.mark.parametrize('heads', [1, 3, 5])
def test_pooling_matches_oracle_and_written_rows_change_nothing(dim, heads):
    spec = helpers.small_layout()
    lay, olay = helpers.product_layout(*spec, device='cuda'), helpers.oracle_layout(*spec)
    x, = helpers.qkv(lay.seq_len, heads, dim, seed=heads, n=1)
    tiles, feats = kernels.gather_and_pool(x.cuda(), lay, None)
    alone, = kernels.pool_seq(x.cuda(), lay, None)
    assert torch.equal(feats, alone)
    want = ot.gather_tiles(x, olay, None)
    assert torch.equal(tiles.cpu(), want)
    pooled = op.pool_tiles(want, olay)
    got = feats.cpu()
    assert torch.equal(got[..., dim:], pooled[..., dim:])
    # 128 fp32 additions of values below 5: 128 * 2^-24 * 5 per element of a mean
    torch.testing.assert_close(got[..., :dim], pooled[..., :dim], rtol=0, atol=128 * 5 * 2.0 ** -24)


def test_head_chunks_keep_the_bits():
    """440 tiles x 28 heads pool as 3,080 items (one wave each); a chunk of
    four heads as 440 (split), and the rows written along with them split."""
    spec = ([(0, (40, 22, 64))], 56320, 56320, '4x2x16')
    lay = helpers.product_layout(*spec, device='cuda')
    x = torch.randn(56320, 28, 128, generator=torch.Generator('cuda').manual_seed(1),
                    device='cuda').to(torch.bfloat16)
    heads = torch.arange(28, device='cuda')
    assert lay.n_tiles * 28 // 4 > 2560 > lay.n_tiles
    whole, = kernels.pool_seq(x, lay, heads)
    parts = torch.cat([kernels.pool_seq(x, lay, h)[0] for h in heads.split(4)])
    assert torch.equal(whole, parts)
    assert torch.equal(whole, kernels.gather_and_pool(x, lay, heads)[1])


@pytest.mark.parametrize('dim', [64, 128])
@pytest.mark.parametrize('second', [False, True])
def test_a_pair_pools_as_its_tensors_alone(dim, second):
    lay = helpers.product_layout(*helpers.small_layout(), device='cuda')
    x, y = (t.cuda() for t in helpers.qkv(lay.seq_len, 5, dim, seed=9, n=2))
    heads = torch.tensor([4, 0, 2, 3, 1], device='cuda')
    for pair in ((x, y), (x[:, 1:], y[:, 1:])):  # whole tensors, and strided views of them
        h = heads if pair[0].shape[1] == 5 else heads[:3] % 4
        got = kernels.pool_seq_pair(*pair, lay, h, second)
        for g, t in zip(got, pair):
            for a, b in zip(g, kernels.pool_seq(t, lay, h, second)):
                assert torch.equal(a, b)
    with pytest.raises(ValueError, match='laid out'):
        kernels.pool_seq_pair(x, y[:, 1:], lay, heads)


@pytest.mark.parametrize('heads', [28, 25])
@pytest.mark.parametrize('second', [False, True])
def test_a_large_pair_pools_as_its_tensors_alone(heads, second):
    """A pair whose launch takes the one-wave form (441 tiles x 7 head groups,
    the last workgroup cut), its tensors alone, and chunks of their heads,
    which take the split form."""
    spec = ([(64, (40, 22, 62))], 54624, 56320, '4x2x16')
    lay = helpers.product_layout(*spec, device='cuda')
    g = torch.Generator('cuda').manual_seed(heads)
    x, y = (torch.randn(56320, heads, 128, generator=g, device='cuda').to(torch.bfloat16) for _ in range(2))
    groups = lay.n_tiles * -(-heads // 4)
    assert 2 * groups >= 2560 > lay.n_tiles and groups % 4
    pair = kernels.pool_seq_pair(x, y, lay, None, second)
    for got, t in zip(pair, (x, y)):
        for a, b in zip(got, kernels.pool_seq(t, lay, None, second)):
            assert torch.equal(a, b)
        few = torch.cat([kernels.pool_seq(t, lay, h)[0] for h in torch.arange(heads, device='cuda').split(4)])
        assert second or torch.equal(got[0], few)


@pytest.mark.parametrize('dim', [64, 128])
@pytest.mark.parametrize('heads', [1, 5, 16])
def test_no_heads_is_every_head_in_order(dim, heads):
    lay = helpers.product_layout(*helpers.small_layout(), device='cuda')
    x, y = (t.cuda() for t in helpers.qkv(lay.seq_len, heads, dim, seed=heads, n=2))
    every = torch.arange(heads, device='cuda')

    def run(h):
        tiles = kernels.gather_tiles(x, lay, h)
        out = torch.full((lay.seq_len + 1, heads, dim), 7., dtype=torch.bfloat16, device='cuda')
        kernels.scatter_tiles_(out, tiles, lay, h)
        return [tiles, out, *kernels.gather_and_pool(x, lay, h, second=True),
                *kernels.pool_seq(x, lay, h), *kernels.pool_seq_pair(x, y, lay, h)[1]]

    for a, b in zip(run(None), run(every)):
        assert torch.equal(a, b)
