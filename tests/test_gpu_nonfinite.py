"""Infinities and NaN in the inputs reach what depends on them, as in plain
arithmetic, and nothing else."""

import math

import pytest
import torch

from miowtion_amd import ops

pytestmark = pytest.mark.gpu

INF, NAN = math.inf, math.nan
H, D = 2, 128


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
