"""Infinities and NaN in the attention walks, the teacher's statistics, the
pooling and the gradients: they reach what depends on them, as in plain
arithmetic, and nothing else."""

import math

import pytest
import torch

from miowtion_amd import kernels
from miowtion_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu

INF, NAN = math.inf, math.nan
H, D = 2, 128
COUNT = torch.tensor([128, 33, 97, 128, 24], dtype=torch.int32)
N = COUNT.numel()
REAL = (torch.arange(128)[None] < COUNT[:, None]).reshape(-1)


def _rand(rows, seed, n=3):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(rows, H, D, generator=g).to(torch.bfloat16) for _ in range(n)]


@pytest.mark.parametrize('used', [65, 100, 321, 447])
def test_dense_infinite_value_gives_infinity(used):
    """One infinite value row gives infinities (its probability is above 0),
    wherever it is but in the last row of a partial step; rows past `used`
    are not looked at."""
    q, k, v = _rand(used + 40, used)
    clean = ops.dense_fwd(q.cuda(), k.cuda(), v.cuda(), used, False)[0].cpu()
    for x in (k, v):
        x[used:] = NAN
    for at in sorted({0, used - 66, used - 64, used - 40, used - 2} & set(range(used))):
        w = v.clone()
        w[at, :, 7] = INF
        out = ops.dense_fwd(q.cuda(), k.cuda(), w.cuda(), used, False)[0].cpu()
        assert (out[:used, :, 7] == INF).all(), at
        rest = torch.arange(D) != 7
        assert torch.equal(out[:used][..., rest], clean[:used][..., rest])


def _walks(q, k, v, mask):
    """The tile-order and the sequence-order forward, in tile order."""
    lists = ops.index_lists(mask.cuda(), (COUNT > 0).cuda(), (COUNT == 128).cuda())
    out, lse = ops.block_sparse_fwd(q.cuda(), k.cuda(), v.cuda(), *lists, COUNT.cuda(), True)
    rows = int(REAL.sum())
    index = (torch.cumsum(REAL.long(), 0) - 1).clamp(min=0)
    buf = torch.zeros(rows + 1, H, D, dtype=torch.bfloat16, device='cuda')
    ops.block_sparse_fwd_seq_kv_(buf, *(x[REAL].contiguous().cuda() for x in (q, k, v)), index.cuda(),
                                 torch.where(REAL, index, rows).cuda(), REAL.int().cuda(),
                                 torch.arange(H, device='cuda'), *lists, COUNT.cuda())
    return [out.cpu()[REAL], buf[:rows].cpu()], lse.cpu()[:, REAL]


def _sparse_case(seed):
    q, k, v = (torch.where(REAL[:, None, None], x, torch.zeros_like(x)) for x in _rand(N * 128, seed))
    mask = torch.eye(N, dtype=torch.bool).repeat(H, 1, 1)
    mask[:, 1:4, 0] = True
    mask[0, 0, 3] = mask[1, 4, 2] = True
    return q, k, v, mask


@pytest.mark.parametrize('tile,row', [(0, 5), (0, 100), (1, 32), (2, 96), (3, 64)])
def test_sparse_only_rows_that_keep_the_tile_see_it(tile, row):
    q, k, v, mask = _sparse_case(row)
    clean, clean_lse = _walks(q, k, v, mask)
    keeps = mask[:, :, tile].repeat_interleave(128, 1)[:, REAL].T  # [rows, H]
    at = tile * 128 + row
    for value in (INF, NAN):
        w = v.clone()
        w[at, :, 7] = value
        for out, want in zip(_walks(q, k, w, mask)[0], clean):
            assert (torch.isfinite(out[..., 7]) == ~keeps).all()
            rest = torch.arange(D) != 7
            assert torch.equal(out[..., rest], want[..., rest])
    w = k.clone()
    w[at, :, 3] = NAN
    outs, lse = _walks(q, w, v, mask)
    for out, want in zip(outs, clean):
        assert torch.isnan(out[keeps]).all() and torch.equal(out[~keeps], want[~keeps])
    assert not torch.isfinite(lse.T[keeps]).any()
    assert torch.equal(lse.T[~keeps], clean_lse.T[~keeps])


@pytest.mark.parametrize('keys', [(0, 1), (0, 32), (0, 64), (0, 128), (32, 96)])
def test_scores_of_minus_infinity_drop_their_keys(keys):
    """Also where a walk begins with them: the rows have no reference until
    later."""
    q, k, v, _ = _sparse_case(keys[1])
    q[REAL, :, 0] = q[REAL, :, 0].abs() + 0.5
    k[keys[0]:keys[1], :, 0] = -INF
    gone = torch.zeros(N * 128, dtype=torch.bool)
    gone[keys[0]:keys[1]] = True
    outs, lse = _walks(q, k, v, torch.ones(H, N, N, dtype=torch.bool))
    ok = REAL & ~gone
    heat, stat_lse = ops.dense_heat(q.cuda(), k.cuda(), None, COUNT.cuda(), torch.arange(N).cuda(), 'sum')
    dense, dense_lse = ops.dense_fwd(q.cuda(), k.cuda(), v.cuda(), 128, True)
    for h in range(H):
        s = q[REAL, h].double() @ k[ok, h].double().T / math.sqrt(D)
        want_lse, want = torch.logsumexp(s, -1), torch.softmax(s, -1) @ v[ok, h].double()
        torch.testing.assert_close(lse[h].double(), want_lse, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(stat_lse[h].cpu()[REAL].double(), want_lse, rtol=1e-5, atol=1e-5)
        for out in outs:  # P and the output round to bf16: 2^-8 each of the largest value
            assert (out[:, h].double() - want).abs().max() <= 2.0 ** -7 * v.abs().max()
        # every real row's probabilities sum to 1; 2e-4 as for any heat of 'sum'
        torch.testing.assert_close(heat[h].sum(-1).cpu(), COUNT.float(), rtol=2e-4, atol=0)
        left = ~gone[:128]
        s = q[:128, h].double() @ k[:128, h][left].double().T / math.sqrt(D)
        if left.any():
            torch.testing.assert_close(dense_lse[:128, h].cpu().double(), torch.logsumexp(s, -1),
                                       rtol=1e-5, atol=1e-5)
            assert (dense[:128, h].cpu().double() - torch.softmax(s, -1) @ v[:128, h][left].double()
                    ).abs().max() <= 2.0 ** -7 * v.abs().max()


@pytest.mark.parametrize('reduce', ['sum', 'max'])
def test_statistics_of_zero_rows_see_a_key_that_is_not_finite(reduce):
    """Whole groups of real rows whose q is zero: 0 times infinity is not 0."""
    q, k, _, _ = _sparse_case(1)
    q[:128] = 0
    q[2 * 128:2 * 128 + 64] = 0
    rows = torch.arange(N).cuda()
    _, clean = ops.dense_heat(q.cuda(), k.cuda(), None, COUNT.cuda(), rows, reduce)
    assert torch.isfinite(clean).all()
    for value in (INF, NAN):
        w = k.clone()
        w[130, 0, 9] = value
        _, lse = ops.dense_heat(q.cuda(), w.cuda(), None, COUNT.cuda(), rows, reduce)
        zero = (q[REAL, 0] == 0).all(-1)
        assert not torch.isfinite(lse[0].cpu()[REAL][zero]).any()
        assert torch.equal(lse[1], clean[1])


@pytest.mark.parametrize('dim', [64, 128])
def test_pooling_forms_agree(dim):
    """The split and the one-wave form of the pooling on infinities and NaN,
    and on a tile whose infinities cancel."""
    spec = ([(0, (40, 22, 64))], 56320, 56320, '4x2x16')
    lay = helpers.product_layout(*spec, device='cuda')
    heads = 28 * 128 // dim
    x = torch.randn(56320, heads, dim, generator=torch.Generator('cuda').manual_seed(2), device='cuda')
    x = x.to(torch.bfloat16)
    for i, value in enumerate((INF, -INF, NAN, -NAN)):
        x[1000 + 7000 * i, :, i] = value
    x[40000, :, 9], x[40001, :, 9] = INF, -INF
    whole, = kernels.pool_seq(x, lay, None)
    assert lay.n_tiles * heads * dim // 512 > 2560
    few = torch.cat([kernels.pool_seq(x, lay, h)[0] for h in torch.arange(heads, device='cuda').split(512 // dim)])
    assert torch.equal(whole.view(torch.int32), few.view(torch.int32))
    mean = whole[..., :dim]
    tiles = kernels.gather_tiles(x[:, :1].contiguous(), lay, None).view(lay.n_tiles, 128, dim).float().sum(1)
    assert torch.equal(torch.isnan(mean[0]), torch.isnan(tiles))
    assert torch.equal(torch.isinf(mean[0]), torch.isinf(tiles))


def test_wide_gradients_keep_them_where_the_narrow_ones_do():
    """dK and dV of a launch of many workgroups (32 keys a wave) against the
    same heads in a launch of few: finite in the same places."""
    spec = helpers.small_layout(grid=(9, 13, 21), shape='2x4x16', text=200, extra=1)
    lay = helpers.product_layout(*spec, device='cuda')
    n, heads = lay.n_tiles, -(-768 // lay.n_tiles)
    g = torch.Generator(device='cuda').manual_seed(3)
    real = lay.slot_valid.bool()
    q, k, v, dout = (torch.where(real[:, None, None], torch.randn(n * 128, heads, 128, generator=g,
                                                                  device='cuda'), 0.0)
                     .to(torch.bfloat16) for _ in range(4))
    mask = (torch.rand(heads, n, n, generator=g, device='cuda') < 0.3) & lay.kv_ok
    mask[:, torch.arange(n), torch.arange(n)] = lay.kv_ok
    mask[:, 2, 1] = False
    dout[3, 0, 5], dout[2 * 128 + 1, 1, 6] = INF, NAN
    pick = [0, 1]

    def grads(sel):
        ins = [t[:, sel].contiguous().requires_grad_(True) for t in (q, k, v)]
        out = kernels.block_sparse_attention(*ins, mask[sel], lay)
        return torch.autograd.grad(out, ins, dout[:, sel].contiguous())

    wide, few = grads(list(range(heads))), grads(pick)
    for name, a, b in zip('qkv', wide, few):
        a, b = a[real][:, pick], b[real]
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), name
        ok = torch.isfinite(b)
        assert not ok.all() and ok.any()
        # finite values: the products' order alone differs (bf16 result, 2^-8)
        d = torch.where(ok, a.float() - b.float(), 0.0)
        assert d.norm() <= 2.0 ** -8 * torch.where(ok, b.float(), 0.0).norm(), name
