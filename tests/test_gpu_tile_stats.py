"""The teacher's statistics pass (dense_heat without the dense output) against
float64 at the edges of its walk: key tiles of every sub-block count (none,
1 .. 32, .. 64, .. 96, .. 128 valid keys), walks of one to several ring slots
with every remainder, query items that do not fill a group of four, query
tiles whose second 64 rows, or all rows, are padding (zero)."""

import math

import pytest
import torch

from miowtion_amd import ops

pytestmark = pytest.mark.gpu

COUNTS = {
    1: [77], 2: [128, 31], 3: [32, 0, 128], 4: [96, 97, 1, 64], 5: [128, 128, 33, 65, 24],
    9: [128, 0, 0, 128, 127, 63, 95, 32, 128],
}


@pytest.mark.parametrize('reduce', ['sum', 'max'])
@pytest.mark.parametrize('n', sorted(COUNTS))
@pytest.mark.parametrize('items', ['all', 'some'])
def test_statistics_match_float64(reduce, n, items):
    g = torch.Generator().manual_seed(n)
    count = torch.tensor(COUNTS[n], dtype=torch.int32)
    real = torch.arange(128)[None] < count[:, None]
    q, k = (torch.randn(n * 128, 3, 128, generator=g).to(torch.bfloat16) for _ in range(2))
    q = q * real.reshape(-1, 1, 1)
    q[:64] = q[:64] * 12  # scores far apart: the reference moves on the way
    rows = torch.arange(n) if items == 'all' else torch.arange(n)[-(n + 1) // 2:]
    heat, lse = ops.dense_heat(q.cuda(), k.cuda(), None, count.cuda(), rows.cuda(), reduce)
    qd = q.double().view(n, 128, 3, 128)[rows].permute(2, 0, 1, 3)           # [3, R, 128, D]
    kd = k.double().view(n * 128, 3, 128).permute(1, 2, 0)[:, None]          # [3, 1, D, N]
    raw = qd @ kd
    s = (raw / math.sqrt(128)).masked_fill(~real.reshape(-1), -math.inf)
    want_lse = torch.logsumexp(s, -1)
    # fp32 scores of 128 products: 1e-5 of a score of up to ~60 covers their rounding
    torch.testing.assert_close(lse.cpu().double(), want_lse.reshape(3, -1), rtol=1e-5, atol=1e-5)
    if reduce == 'sum':
        p = torch.exp(s - want_lse[..., None]).view(3, rows.numel(), 128, n, 128).sum(-1)
        want = torch.where(real[rows][None, :, :, None], p, 0.0).sum(2)
        torch.testing.assert_close(heat.cpu().double(), want, rtol=2e-4, atol=1e-7)
    else:
        top = raw.masked_fill(~real.reshape(-1), -math.inf).view(3, rows.numel(), 128, n, 128).amax(-1)
        top = top.to(torch.bfloat16).double() / math.sqrt(128)               # rounded before the scale
        p = torch.exp(top - want_lse[..., None])
        want = torch.where(real[rows][None, :, :, None], p, 0.0).amax(2)
        # a raw maximum next to a bf16 rounding boundary may round the other way: 2^-8 of a
        # score of up to ~60
        torch.testing.assert_close(heat.cpu().double(), want, rtol=60 * 2.0 ** -8, atol=1e-7)
