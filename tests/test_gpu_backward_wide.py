"""dK and dV of launches of many (head, key tile) workgroups, which take 32
keys a wave: against the oracle on two heads, and against the same heads in a
launch of few workgroups. Key tiles with every kind of fill (3 to 128 valid
keys: one, two and four key groups, full and cut), dense output gradients,
gradients that are zero on padding rows (steps left out, steps whose upper
half is), and an LSE gradient."""

import pytest
import torch

from miowtion_amd import kernels
from oracle import attention as oa
from tests import helpers

pytestmark = pytest.mark.gpu

ITEMS = 768  # from here on a launch takes 32 keys a wave, unless few walks are much longer
RESIDENT = 512  # workgroups at once; 2/3 of them is where the longest walk decides


def _heads(lay, n):
    """Enough heads that the global key tiles' walks (`front` of them, over
    every query tile) do not put the launch to the 16-key form."""
    front = n - lay.n_video_tiles
    return max(-(-ITEMS // n), -(-2 * RESIDENT // (3 * (2 * front + 1))))


LAYOUTS = [dict(grid=(3, 9, 11), shape='2x8x8', text=5, extra=3),
           dict(grid=(9, 13, 21), shape='2x4x16', text=200, extra=1)]


@pytest.mark.parametrize('kind', range(len(LAYOUTS)))
@pytest.mark.parametrize('grad', ['dense', 'layer', 'lse'])
def test_wide_launch(kind, grad):
    spec = helpers.small_layout(**LAYOUTS[kind])
    lay, olay = helpers.product_layout(*spec, device='cuda'), helpers.oracle_layout(*spec)
    n, heads = lay.n_tiles, _heads(lay, lay.n_tiles)
    rows = n * 128
    g = torch.Generator(device='cuda').manual_seed(10 * kind)
    real = lay.slot_valid.bool()[:, None, None]
    q, k, v = (torch.where(real, torch.randn(rows, heads, 128, generator=g, device='cuda'), 0.0)
               .to(torch.bfloat16) for _ in range(3))
    mask = (torch.rand(heads, n, n, generator=g, device='cuda') < 0.4) & lay.kv_ok
    mask[:, torch.arange(n), torch.arange(n)] = lay.kv_ok
    mask[:, 1, 0] = False
    mask[-1, :, 0] = False  # a key tile that no query tile keeps
    dout = torch.randn(rows, heads, 128, generator=g, device='cuda').to(torch.bfloat16)
    if grad == 'layer':
        dout = torch.where(real, dout, torch.zeros_like(dout))
    dlse = torch.randn(heads, rows, generator=g, device='cuda') if grad == 'lse' else None

    def grads(sel):
        ins = [t[:, sel].contiguous().requires_grad_(True) for t in (q, k, v)]
        out, lse = kernels.block_sparse_attention(*ins, mask[sel], lay, return_lse=True)
        if dlse is None:
            return torch.autograd.grad(out, ins, dout[:, sel].contiguous())
        return torch.autograd.grad((out, lse), ins, (dout[:, sel].contiguous(), dlse[sel]))

    pick = [0, heads - 1]
    assert heads * n >= ITEMS > len(pick) * n
    wide, few = grads(list(range(heads))), grads(pick)
    want = oa.block_sparse_attention_grads(
        *(t[:, pick].cpu() for t in (q, k, v)), mask[pick].cpu(), olay.valid_count,
        dout[:, pick].cpu().float(), None if dlse is None else dlse[pick].cpu())
    assert not torch.equal(wide[1][:, pick], few[1])  # the other form's order of sums
    for name, a, b, w in zip('qkv', wide, few, want):
        a, b = a[:, pick].cpu().float(), b.cpu().float()
        # the products take bf16 P and dS (2^-9 rms each) and the result rounds to bf16
        assert (a - w).norm() <= 1e-2 * w.norm(), name
        assert (a - b).norm() <= 2.0 ** -8 * b.norm(), name
        assert (a - w).norm() <= 1.02 * (b - w).norm(), name  # no less precise than few
    pad = ~real[:, 0, 0].cpu()
    assert (wide[1].cpu()[pad] == 0).all() and (wide[2].cpu()[pad] == 0).all()


@pytest.mark.parametrize('text,keep,wide', [(500, 0.05, False), (500, 1.0, True), (40, 0.1, False),
                                            (40, 1.0, True)])
def test_long_walks_take_the_form_of_few_workgroups(text, keep, wide):
    """Global key tiles, which every query tile keeps, beside video tiles of
    few: the 16-key form, so the bits of a launch of few heads; beside video
    tiles as long as theirs, 32 keys a wave."""
    spec = helpers.small_layout(grid=(9, 26, 42), shape='2x4x16', text=text, extra=1)
    lay = helpers.product_layout(*spec, device='cuda')
    n, heads = lay.n_tiles, -(-ITEMS // lay.n_tiles)
    front = n - lay.n_video_tiles
    assert front > 0 and 3 * heads * (2 * front + 1) < 2 * RESIDENT
    g = torch.Generator(device='cuda').manual_seed(text)
    q, k, v, dout = (torch.randn(n * 128, heads, 128, generator=g, device='cuda').to(torch.bfloat16)
                     * lay.slot_valid[:, None, None].to(torch.bfloat16) for _ in range(4))
    mask = torch.rand(heads, n, n, generator=g, device='cuda') < keep
    mask[:, torch.arange(n), torch.arange(n)] = True
    mask[:, :, lay.n_video_tiles:] = True
    mask[:, lay.n_video_tiles:] = True
    mask &= lay.kv_ok
    walks = mask.sum(1).flatten()
    assert (3 * walks.sum() >= 2 * RESIDENT * walks.max()) == wide

    def grads(sel):
        ins = [t[:, sel].contiguous().requires_grad_(True) for t in (q, k, v)]
        out = kernels.block_sparse_attention(*ins, mask[sel], lay)
        return torch.autograd.grad(out, ins, dout[:, sel].contiguous())

    pick = [0, heads - 1]
    many, few = grads(list(range(heads))), grads(pick)
    assert torch.equal(many[0][:, pick], few[0])
    for a, b in zip(many[1:], few[1:]):
        a, b = a[:, pick], b
        assert torch.equal(a, b) != wide
        assert (a.float() - b.float()).norm() <= 2.0 ** -8 * b.float().norm()
