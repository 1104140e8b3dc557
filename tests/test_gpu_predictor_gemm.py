"""The predictor's embedding product at the edges of its tiles and of its
weight loads, against the same product in float64: k below, at and past a
32-k block; n_out that is and is not whole groups of eight columns; weights
whose start is not 16-byte aligned; every weight format; a head id outside
the weights (its embedding is the residual alone)."""

import pytest
import torch

from miowtion_amd import ops

pytestmark = pytest.mark.gpu


def _weights(fmt, heads, k, n, offset, g):
    """([heads, k, n] values whose storage starts `offset` elements in, scale,
    the float64 values the product uses)."""
    w = torch.randn(heads, k, n, generator=g) * 0.05
    scale = None
    if fmt == 'fp8':
        scale = w.abs().amax((1, 2)) / 448
        w = (w / scale[:, None, None]).to(torch.float8_e4m3fn)
        used = (w.float() * scale[:, None, None]).to(torch.bfloat16).double()
    else:
        w = w.to(torch.bfloat16 if fmt == 'bf16' else torch.float32)
        used = w.double()
    raw = w.contiguous().view(torch.uint8).flatten()
    size = raw.numel() // w.numel()
    buf = torch.zeros(raw.numel() + 64, dtype=torch.uint8, device='cuda')
    buf[offset * size:offset * size + raw.numel()] = raw.cuda()
    values = buf[offset * size:offset * size + raw.numel()].view(w.dtype).view(heads, k, n)
    return values, None if scale is None else scale.cuda(), used


@pytest.mark.parametrize('fmt', ['fp8', 'bf16', 'fp32'])
@pytest.mark.parametrize('m,k,n,offset', [
    (1, 4, 8, 0), (65, 36, 16, 0), (64, 384, 128, 0), (130, 384, 64, 0), (7, 100, 72, 0),
    (33, 384, 12, 0), (33, 64, 128, 4), (9, 32, 8, 8),
])
def test_embedding_matches_float64(fmt, m, k, n, offset):
    g = torch.Generator().manual_seed(m * 1000 + k + n)
    feats = torch.randn(3, m, k, generator=g)
    values, scale, used = _weights(fmt, 4, k, n, offset, g)
    heads = torch.tensor([2, 9, 0])
    residual = k >= n
    got = ops.predictor_embed(feats.cuda(), values, scale, heads.cuda(), residual).cpu().double()
    used = torch.stack([used[2], torch.zeros_like(used[0]), used[0]])
    want = feats.double() @ used
    size = feats.double().abs() @ used.abs()
    if residual:
        want = want + feats[..., :n].double()
        size = size + feats[..., :n].double().abs()
    # k + 1 roundings of fp32 sums, each at most 2^-24 of the sum of magnitudes
    assert ((got - want).abs() <= (k + 1) * 2.0 ** -24 * size + 1e-30).all()


@pytest.mark.parametrize('fmt', ['fp8', 'bf16', 'fp32'])
@pytest.mark.parametrize('m,k,n', [(70, 384, 128), (9, 64, 16), (5, 30, 8), (5, 32, 12)])
def test_a_pair_embeds_as_its_products_alone(fmt, m, k, n):
    g = torch.Generator().manual_seed(m + k)
    feats = [torch.randn(3, m, k, generator=g).cuda() for _ in range(2)]
    (wa, sa, _), (wb, sb, _) = (_weights(fmt, 4, k, n, 0, g) for _ in range(2))
    heads = torch.tensor([3, 0, 7], device='cuda')
    got = ops.predictor_embed_pair(*feats, wa, wb, sa, sb, heads, k >= n)
    assert torch.equal(got[0], ops.predictor_embed(feats[0], wa, sa, heads, k >= n))
    assert torch.equal(got[1], ops.predictor_embed(feats[1], wb, sb, heads, k >= n))


def test_a_pair_of_more_heads_than_one_launch_takes():
    g = torch.Generator().manual_seed(1)
    feats = [torch.randn(32768, 1, 4, generator=g).cuda() for _ in range(2)]
    (wa, sa, _), (wb, sb, _) = (_weights('bf16', 4, 4, 8, 0, g) for _ in range(2))
    heads = torch.randint(0, 4, (32768,), generator=g).cuda()
    got = ops.predictor_embed_pair(*feats, wa, wb, sa, sb, heads, False)
    assert torch.equal(got[0], ops.predictor_embed(feats[0], wa, sa, heads, False))
    assert torch.equal(got[1], ops.predictor_embed(feats[1], wb, sb, heads, False))
