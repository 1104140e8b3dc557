"""The pipelined attention walks against float64 where the pipeline fills,
drains and branches: walks of one to several steps, odd and even; key tiles
with every kind of ragged end; query tiles whose rows fill one, two, three or
four waves; scores that jump far past a row's first sub-block (the reference
is raised mid-walk, also in the last sub-block); and the sequence-order entry,
bit for bit against the tile-order one."""

import math

import pytest
import torch

from miowtion_amd import ops

pytestmark = pytest.mark.gpu

H, D = 2, 128
COUNTS = {
    1: [128], 2: [24, 128], 3: [32, 96, 1], 4: [128, 33, 64, 97],
    6: [128, 24, 32, 96, 128, 65], 11: [128, 128, 24, 1, 96, 31, 64, 128, 33, 127, 128],
}


def _case(n, jump):
    g = torch.Generator().manual_seed(100 * n + jump)
    count = torch.tensor(COUNTS[n], dtype=torch.int32)
    real = (torch.arange(128)[None] < count[:, None]).reshape(-1, 1, 1)
    q, k, v = (torch.where(real, torch.randn(n * 128, H, D, generator=g), 0.0).to(torch.bfloat16)
               for _ in range(3))  # padding rows +0, as the gather writes them
    if jump:  # later tiles and, within a tile, later keys score ever higher
        grow = 1 + 3 * torch.arange(n * 128).float() / 128
        k = (k.float() * grow[:, None, None]).to(torch.bfloat16)
    mask = torch.rand(H, n, n, generator=g) < 0.6
    mask[:, torch.arange(n), torch.arange(n)] = True
    if n > 3:
        mask[0, 2] = False  # a query tile that keeps nothing
        mask[1, 3] = True
    return count, q, k, v, mask


def _exact(q, k, v, mask, count):
    n = count.numel()
    real = (torch.arange(128)[None] < count[:, None]).reshape(-1)
    out, lse = torch.zeros(n * 128, H, D).double(), torch.full((H, n * 128), -math.inf).double()
    for h in range(H):
        ok = mask[h].repeat_interleave(128, 0).repeat_interleave(128, 1) & real[None]
        s = (q[:, h].double() @ k[:, h].double().T / math.sqrt(D)).masked_fill(~ok, -math.inf)
        lse[h] = torch.logsumexp(s, -1)
        out[:, h] = torch.nan_to_num(torch.softmax(s, -1)) @ v[:, h].double()
    return out, lse


def _close(out, lse, want, want_lse, v):
    # P and the output round to bf16 (7 fraction bits: 2^-8 each, of the largest value averaged)
    off = out.cpu().double() - want
    assert off.abs().max() <= 2.0 ** -7 * v.abs().max().item()
    # over all values the two roundings are independent, each uniform in a relative 2^-8 at most:
    # 2^-8 / sqrt(3) rms each
    assert off.norm() <= math.sqrt(2 / 3) * 2.0 ** -8 * want.norm()
    if lse is not None:
        torch.testing.assert_close(lse.cpu().double(), want_lse, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize('jump', [0, 1])
@pytest.mark.parametrize('n', sorted(COUNTS))
def test_sparse_walk_and_sequence_order(n, jump):
    count, q, k, v, mask = _case(n, jump)
    kv_ok, full = count > 0, count == 128
    lists = ops.index_lists(mask.cuda(), kv_ok.cuda(), full.cuda())
    out, lse = ops.block_sparse_fwd(q.cuda(), k.cuda(), v.cuda(), *lists, count.cuda(), True)
    _close(out, lse, *_exact(q, k, v, mask, count), v)
    # the rows scattered over a sequence, read and written through the indices
    real = (torch.arange(128)[None] < count[:, None]).reshape(-1)
    rows = int(real.sum())
    perm = torch.randperm(rows, generator=torch.Generator().manual_seed(n))
    index = torch.zeros(n * 128, dtype=torch.int64)
    index[real] = perm
    scatter = torch.where(real, index, rows)
    seq = [torch.zeros(rows, H, D, dtype=torch.bfloat16) for _ in range(3)]
    for s, x in zip(seq, (q, k, v)):
        s[perm] = x[real]
    buf = torch.full((rows + 1, H, D), 7.0, dtype=torch.bfloat16, device='cuda')
    ops.block_sparse_fwd_seq_kv_(buf, *(s.cuda() for s in seq), index.cuda(), scatter.cuda(),
                                 real.int().cuda(), torch.arange(H, device='cuda'), *lists, count.cuda())
    assert torch.equal(buf[perm.cuda()], out[real.cuda()])
    assert (buf[rows] == 7.0).all()


def test_zero_query_rows_that_are_stored():
    """Whole 32-row groups of real rows whose q is zero, beside padding
    groups, in sequence order: stored rows are computed, dropped ones not."""
    for groups in ([1, 0, 0, 0], [0, 1, 0, 0], [1, 0, 1, 0], [0, 0, 0, 0], [1, 0, 0, 1]):
        for valid in (128, 96, 64, 40):
            count = torch.tensor([valid, 128], dtype=torch.int32)
            g = torch.Generator().manual_seed(valid)
            real = (torch.arange(128)[None] < count[:, None]).reshape(-1)
            q, k, v = (torch.where(real[:, None, None], torch.randn(256, H, D, generator=g), 0.0)
                       .to(torch.bfloat16) for _ in range(3))
            keep = torch.tensor(groups).repeat_interleave(32).repeat(2).bool()
            q = torch.where(keep[:, None, None], q, 0.0).to(torch.bfloat16)
            mask = torch.ones(H, 2, 2, dtype=torch.bool)
            lists = ops.index_lists(mask.cuda(), (count > 0).cuda(), (count == 128).cuda())
            want, _ = _exact(q, k, v, mask, count)
            index = torch.cumsum(real.long(), 0) - 1
            rows = int(real.sum())
            buf = torch.zeros(rows + 1, H, D, dtype=torch.bfloat16, device='cuda')
            ops.block_sparse_fwd_seq_kv_(
                buf, *(x[real].contiguous().cuda() for x in (q, k, v)), index.clamp(min=0).cuda(),
                torch.where(real, index, rows).cuda(), real.int().cuda(),
                torch.arange(H, device='cuda'), *lists, count.cuda())
            _close(buf[:rows], None, want[real], None, v)


@pytest.mark.parametrize('used', [1, 31, 33, 63, 64, 65, 96, 127, 128, 129, 191, 193, 256, 257, 321, 448])
@pytest.mark.parametrize('jump', [0, 1])
def test_dense_walk(used, jump):
    g = torch.Generator().manual_seed(used + jump)
    q, k, v = (torch.randn(used + 5, H, D, generator=g).to(torch.bfloat16) for _ in range(3))
    if jump:
        k = (k.float() * (1 + torch.arange(used + 5).float() / 32)[:, None, None]).to(torch.bfloat16)
    out, lse = ops.dense_fwd(q.cuda(), k.cuda(), v.cuda(), used, True)
    want, want_lse = torch.zeros(used + 5, H, D).double(), torch.zeros(used + 5, H).double()
    for h in range(H):
        s = q[:used, h].double() @ k[:used, h].double().T / math.sqrt(D)
        want_lse[:used, h] = torch.logsumexp(s, -1)
        want[:used, h] = torch.softmax(s, -1) @ v[:used, h].double()
    _close(out, lse, want, want_lse, v)
