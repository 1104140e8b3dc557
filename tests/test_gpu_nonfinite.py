"""Infinities and NaN in the inputs reach what depends on them, as in plain
arithmetic, and nothing else."""

import math

import pytest
import torch

from miowtion_amd import ops

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


def _sparse_case(seed):
    q, k, v = (torch.where(REAL[:, None, None], x, torch.zeros_like(x)) for x in _rand(N * 128, seed))
    mask = torch.eye(N, dtype=torch.bool).repeat(H, 1, 1)
    mask[:, 1:4, 0] = True
    mask[0, 0, 3] = mask[1, 4, 2] = True
    return q, k, v, mask


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
