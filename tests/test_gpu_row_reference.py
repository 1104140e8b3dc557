"""The attention walks take a row's probabilities relative to the maximum of
its first 64 keys, raised once a later score is 2^8 above it: a key that
dominates its row then has the probability 1, which bf16 holds exactly, and
the output's own rounding is all that is left of the error."""

import math

import pytest
import torch

from miowtion_amd import ops

pytestmark = pytest.mark.gpu

H, D, N = 2, 128, 256


def _case(at, seed):
    """Rows whose score is 0 for every key but key `at`, where it is 10 to
    11.5 above (log2): less than 6 % of the row's mass is on other keys, and
    the ratio of the two probabilities is not a power of two."""
    g = torch.Generator().manual_seed(seed)
    k = torch.zeros(N, H, D)
    k[at, :, 0] = 8.0
    q = torch.zeros(N, H, D)
    q[:, :, 0] = (10 + 1.5 * torch.rand(N, H, generator=g)) * math.log(2.0) * math.sqrt(D) / 8.0
    v = torch.randn(N, H, D, generator=g)
    return [x.to(torch.bfloat16) for x in (q, k, v)]


def _check(out, q, k, v):
    for h in range(H):
        p = torch.softmax(q[:, h].double() @ k[:, h].double().T / math.sqrt(D), -1)
        want = p @ v[:, h].double()
        rest = 1 - p.amax(-1, keepdim=True)
        # half a unit of the output's bf16, and P's rounding (2^-8 at most) on the mass of the
        # other keys alone; fp32 scores and sums 1e-5
        half_unit = 2.0 ** (torch.floor(torch.log2(want.abs().clamp(min=1e-30))) - 8)
        bound = half_unit + 2.0 ** -8 * rest * v.abs().max() + 1e-5
        assert ((out[:, h].cpu().double() - want).abs() <= bound).all()


# keys of the first sub-block, of the second, and of later steps (the reference is raised)
@pytest.mark.parametrize('at', [3, 40, 63, 70, 127, 133, 250])
def test_dominating_key_is_not_rounded(at):
    q, k, v = _case(at, at)
    n = N // 128
    count = torch.full((n,), 128, dtype=torch.int32)
    lists = ops.index_lists(torch.ones(H, n, n, dtype=torch.bool).cuda(), (count > 0).cuda(),
                            (count == 128).cuda())
    _check(ops.block_sparse_fwd(q.cuda(), k.cuda(), v.cuda(), *lists, count.cuda(), False)[0], q, k, v)
    _check(ops.dense_fwd(q.cuda(), k.cuda(), v.cuda(), N, False)[0], q, k, v)
