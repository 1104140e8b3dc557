"""The work that users of this package have it do, as measurable cases.

Every case calls public entry points only, on inputs that stand for a video
diffusion transformer's attention: q, k and v are unit noise, and q and k
share a smooth field over the (t, h, w) grid, so that a token attends to its
neighbourhood more than to the rest, as it does after training.

Kinds of case:
  layer    one sparse attention layer as a model calls it (SparseStudent):
           pooling, predictor, top-k, block lists, block-sparse attention in
           sequence order; with global text rows, tiled reference images, two
           tile shapes, second-order predictor or compensation where asked
  sparse   the block-sparse forward on prebuilt lists (a mask kept over steps)
  train    block-sparse attention forward and backward on tile-ordered q, k, v
  dense    dense attention with its LSE (the teacher, and dense layers)
  teacher  the teacher-masked layer (OracleStudent): dense statistics, block
           heat, top-k on it, block-sparse attention
  permute  permutation into tiles with pooling, and back
"""

from __future__ import annotations

import math

import numpy as np
import torch

from miowtion_amd import attention as pa
from miowtion_amd import kernels
from miowtion_amd import mask as pm
from miowtion_amd import plan as pplan
from miowtion_amd import predictor as pp
from miowtion_amd import tiling as pt

D = 128
TILE = 128
# what an optional field of a case is when it is absent
DEFAULTS = dict(text=0, ref='', ref_keep=0.3, shapes='1x8x16', keep=0.1, fp8=True, rank=0,
                count=False, comp=False, lse_grad=False)


def listed() -> list[dict]:
    return [
        # the smallest layer: a four-frame preview, where launches and host
        # work are all that counts
        dict(name='layer_preview', kind='layer', grid='4x16x16', heads=8, shapes='2x8x8', keep=0.5),
        # an odd short clip behind a text prompt, with one tiled reference
        # image and the full predictor (second-order and count terms, bf16
        # weights): every option of the selection at once
        dict(name='layer_reference', kind='layer', grid='13x24x42', heads=24, shapes='8x4x4', keep=0.2,
             text=333, ref='1x24x42', ref_keep=0.4, fp8=False, rank=16, count=True),
        # the layer of a five-second 16:9 clip, one tile shape, fp8 predictor:
        # the ordinary inference call
        dict(name='layer_16x9', kind='layer', grid='37x30x52', heads=48, shapes='1x8x16', keep=0.1),
        # the same length in 9:16 with a tile shape per head and less sparsity
        dict(name='layer_9x16_two_shapes', kind='layer', grid='37x52x30', heads=48,
             shapes='1x8x16,4x4x8', keep=0.2),
        # the ordinary clip with the dropped tiles compensated
        dict(name='layer_compensated', kind='layer', grid='37x24x42', heads=56, shapes='2x8x8',
             keep=0.1, comp=True),
        # the longest clip, with 2,048 text and audio rows that stay dense
        dict(name='layer_long', kind='layer', grid='102x30x52', heads=48, shapes='1x8x16', keep=0.05,
             text=2048),
        # the kernel alone on uniform random block lists, as the benchmark
        # times it: lists kept over several denoising steps
        dict(name='sparse_16x9', kind='sparse', grid='37x30x52', heads=48, shapes='1x8x16', keep=0.1),
        # a training step of the layer: the output gradient comes back through
        # the scatter, so it is zero on padding rows
        dict(name='train_16x9', kind='train', grid='37x30x52', heads=48, shapes='1x8x16', keep=0.1),
        # a short ragged clip with text rows in training, with an LSE gradient
        dict(name='train_short', kind='train', grid='8x12x20', heads=24, shapes='4x8x4', keep=0.3,
             text=360, lse_grad=True),
        # dense attention with its LSE: dense layers and the teacher
        dict(name='dense_16x9', kind='dense', grid='37x30x52', heads=48),
        # the teacher-masked layer used to fit the predictor, by block mass
        dict(name='teacher_16x9', kind='teacher', grid='37x24x42', heads=56, shapes='8x4x4', keep=0.1),
        # the permutations alone: into tiles with pooling, and back
        dict(name='permute_16x9', kind='permute', grid='37x30x52', heads=48, shapes='1x8x16'),
    ]


def draw(rng) -> dict:
    top = max(work(c)['flops'] for c in listed())
    while True:
        kind = rng.choice(['layer', 'layer', 'layer', 'sparse', 'train', 'dense', 'teacher', 'permute'])

        def log(lo, hi):
            return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

        grid = (log(2, 102), log(8, 52), log(8, 52))
        case = dict(kind=kind, grid=_text(grid), heads=rng.choice([3, 8, 16, 24, 40, 48, 56]),
                    text=rng.choice([0, 0, rng.randint(1, 2048)]))
        if kind != 'dense':
            shapes = [s for s in pt.candidate_shapes(grid) if s.padding_ratio(grid) <= 0.4]
            shapes = shapes or [pt.least_padding_shape(grid)]
            n = 2 if kind in ('layer', 'teacher') and len(shapes) > 1 and rng.random() < 0.4 else 1
            case['shapes'] = ','.join(str(s) for s in rng.sample(shapes, n))
            case['keep'] = round(math.exp(rng.uniform(math.log(0.05), math.log(0.5))), 3)
        if kind in ('layer', 'train') and rng.random() < 0.25:
            case['ref'] = _text((1, grid[1], grid[2]))
            case['ref_keep'] = round(rng.uniform(0.2, 1.0), 2)
        if kind == 'layer':
            case['fp8'] = rng.random() < 0.6
            case['rank'] = rng.choice([0, 0, 16])
            case['count'] = rng.random() < 0.3
            case['comp'] = rng.random() < 0.2
        if kind == 'train':
            case['lse_grad'] = rng.random() < 0.3
        rows = _used(case)
        if rows > 161168 or rows * case['heads'] > 161168 * 48 or work(case)['flops'] > top:
            continue
        # training and teacher passes cost more per product than a forward
        if kind in ('train', 'teacher') and 3 * work(case)['flops'] > top:
            continue
        return case


# ---------------------------------------------------------------------------
# Sizes


def _text(grid) -> str:
    return 'x'.join(str(g) for g in grid)


def _grid(text: str) -> tuple:
    return tuple(int(g) for g in text.split('x'))


def _get(case: dict, key: str):
    return case.get(key, DEFAULTS[key])


def _spans(case: dict) -> list[tuple]:
    """(start, grid) of the tiled spans, references first; the text rows come
    before them."""
    at = _get(case, 'text')
    out = []
    for g in ([_grid(case['ref'])] if _get(case, 'ref') else []) + [_grid(case['grid'])]:
        out.append((at, g))
        at += g[0] * g[1] * g[2]
    return out


def _used(case: dict) -> int:
    start, g = _spans(case)[-1]
    return start + g[0] * g[1] * g[2]


def _seq_len(case: dict) -> int:
    return -(-_used(case) // 64) * 64


def _shape_of_head(case: dict) -> list[int]:
    """The tile shape index of each head."""
    n = len(_get(case, 'shapes').split(','))
    return [h % n for h in range(case['heads'])]


def work(case: dict) -> dict:
    """Real (query row, key row) pairs of the kept blocks; every input read
    once and every output written once."""
    used, heads, kind = _used(case), case['heads'], case['kind']
    t, h, w = _grid(case['grid'])
    target, text = t * h * w, _get(case, 'text')
    row = heads * D * 2
    if kind == 'permute':
        n = -(-used // TILE)
        return {'bytes': float(4 * used * row + n * heads * 3 * D * 4), 'flops': float(2 * used * heads * D)}
    dense = 4.0 * used * used * heads * D
    if kind == 'dense':
        return {'bytes': float(4 * used * row + 4 * used * heads), 'flops': dense}
    ideal = -(-target // TILE)
    kept = 0.0  # kept target keys of a query row, averaged over the shapes
    shapes = _get(case, 'shapes').split(',')
    for st, sh, sw in map(_grid, shapes):
        n = -(-t // st) * -(-h // sh) * -(-w // sw)
        kept += min(1.0, _get(case, 'keep') * ideal * ideal / n / n) * target / len(shapes)
    kept += text
    if _get(case, 'ref'):
        rt, rh, rw = _grid(case['ref'])
        kept += min(1.0, case['ref_keep']) * rt * rh * rw
    video = used - text
    pairs = video * min(kept, used) + text * used
    flops = 4.0 * pairs * heads * D
    moved = 4 * used * row
    if kind == 'layer':
        n = -(-used // TILE)
        flops += 2.0 * n * 2 * 3 * D * D * heads + 2.0 * n * n * D * heads
        moved += 2 * 3 * D * D * heads * (1 if _get(case, 'fp8') else 2)
        if _get(case, 'comp'):
            flops += 4.0 * used * n * D * heads
    elif kind == 'train':
        flops *= 3.5  # two products forward, five backward
        moved = 8 * used * row + 4 * used * heads
    elif kind == 'teacher':
        flops += dense / 2
    return {'bytes': float(moved), 'flops': flops}


def tolerance(case: dict):
    """About four times what the path shows against `exact` (relative
    2-norm): bf16 outputs and gradients 2.1e-3 to 2.7e-3, an fp32 LSE 6e-8,
    pooled features 2e-9 (the permuted rows themselves are copies)."""
    if case['kind'] == 'permute':
        return {'rel': 1e-6}
    return {'rel': 1e-2}


# ---------------------------------------------------------------------------
# Inputs


def _generator(case: dict, seed: int) -> torch.Generator:
    return torch.Generator(device='cuda').manual_seed(1000003 * seed + 17 * _used(case) + case['heads'])


def _field(case: dict, g: torch.Generator) -> torch.Tensor:
    """[seq_len, H, D] smooth in t, h and w on the spans, 0 elsewhere: per
    axis, unit noise on a coarse line, interpolated."""
    heads = case['heads']
    out = torch.zeros(_seq_len(case), heads, D, device='cuda')
    for start, grid in _spans(case):
        part = torch.zeros(*grid, heads * D, device='cuda')
        for axis, n in enumerate(grid):
            line = torch.randn(1, heads * D, max(2, n // 6 + 1), generator=g, device='cuda')
            line = torch.nn.functional.interpolate(line, size=n, mode='linear', align_corners=True)
            shape = [1, 1, 1, heads * D]
            shape[axis] = n
            part += line[0].T.reshape(shape)
        rows = grid[0] * grid[1] * grid[2]
        out[start:start + rows] = part.reshape(rows, heads, D)
    return out * (0.5 / math.sqrt(3.0))


def _qkv(case: dict, g: torch.Generator) -> list[torch.Tensor]:
    """q, k, v [seq_len, H, D] bf16, rows past `used` zero."""
    field = _field(case, g)
    used = _used(case)
    out = []
    for i in range(3):
        x = torch.randn(field.shape, generator=g, device='cuda')
        if i < 2:
            x += field
        x[used:] = 0
        out.append(x.to(torch.bfloat16))
    return out


def _weights(case: dict, g: torch.Generator) -> dict:
    """Predictor weights: name -> (resident values, scale or None)."""
    heads, rank = case['heads'], _get(case, 'rank')
    shapes = dict(proj_q=(3 * D, D), proj_k=(3 * D, D))
    if rank:
        shapes.update(so_q=(D, rank), so_k=(D, rank))
    out = {}
    for name, (a, b) in shapes.items():
        x = torch.randn(heads, a, b, generator=g, device='cuda') * 0.02
        if _get(case, 'fp8'):
            scale = (x.abs().amax((1, 2)) / 448.0).clamp(min=1e-30)
            out[name] = ((x / scale[:, None, None]).to(torch.float8_e4m3fn), scale)
        else:
            out[name] = (x.to(torch.bfloat16), None)
    return out


def _gain(case: dict) -> torch.Tensor:
    return torch.linspace(0.1, 0.5, case['heads'], device='cuda')


def _scores(case: dict, n: int, g: torch.Generator) -> torch.Tensor:
    """Uniform tile scores of the kinds that take a mask."""
    return torch.rand(case['heads'], n, n, generator=g, device='cuda')


def prepare(case: dict, seed: int) -> dict:
    kind, heads = case['kind'], case['heads']
    used, seq_len = _used(case), _seq_len(case)
    g = _generator(case, seed)
    q, k, v = _qkv(case, g)
    if kind == 'dense':
        return dict(kind=kind, q=q, k=k, v=v, used=used)
    spans = _spans(case)
    shapes = [pt.TileShape.parse(s) for s in _get(case, 'shapes').split(',')]
    config = pa.VedaConfig(target_budget=pm.Budget(ratio=_get(case, 'keep')),
                           ref_budget=pm.Budget(ratio=_get(case, 'ref_keep')) if _get(case, 'ref') else None,
                           tile_conditions=bool(_get(case, 'ref')),
                           zero_order_compensation=_get(case, 'comp'))
    packed = pa.PackedLayout(tuple(pa.VideoSpan(s, gr) for s, gr in spans), used, seq_len)
    clip = pa.ClipTiling(packed, config, 'cuda')
    if kind in ('layer', 'teacher'):
        plan = pplan.TilePlan('clip', spans[-1][1], shapes, [_shape_of_head(case)])
        for s in shapes:
            clip.get(s)
        if kind == 'teacher':
            student = pa.OracleStudent(clip, plan)
        else:
            w = {name: pp.ProjWeight(*x) for name, x in _weights(case, g).items()}
            layer = pp.LayerPredictor(w['proj_q'], w['proj_k'], w.get('so_q'), w.get('so_k'),
                                      _gain(case) if _get(case, 'count') else None)
            student = pa.SparseStudent(clip, plan, pp.TileScorePredictor([layer]))
        return dict(kind=kind, q=q, k=k, v=v, student=student)
    layout = clip.get(shapes[0])
    if kind == 'permute':
        back = torch.zeros(seq_len + 1, heads, D, dtype=torch.bfloat16, device='cuda')
        return dict(kind=kind, x=k, layout=layout, back=back)
    qt, kt, vt = (kernels.gather_tiles(x, layout, None) for x in (q, k, v))
    selection = pm.select_video_blocks(_scores(case, layout.n_video_tiles, g), layout, clip.blocks(layout))
    mask = pm.dense_block_mask(selection, layout)
    if kind == 'sparse':
        return dict(kind=kind, q=qt, k=kt, v=vt, lists=kernels.index_lists(mask, layout), layout=layout)
    dout, dlse = _out_grads(case, layout.n_tiles, g)
    dout = dout * layout.slot_valid[:, None, None].to(dout.dtype)
    return dict(kind=kind, q=qt.requires_grad_(), k=kt.requires_grad_(), v=vt.requires_grad_(), mask=mask,
                layout=layout, dout=dout, dlse=dlse)


def _out_grads(case: dict, n: int, g: torch.Generator):
    """Gradients of the output [n * 128, H, D] bf16 and, where asked, the LSE."""
    dout = torch.randn(n * TILE, case['heads'], D, generator=g, device='cuda').to(torch.bfloat16)
    dlse = None
    if _get(case, 'lse_grad'):
        dlse = torch.randn(case['heads'], n * TILE, generator=g, device='cuda') * 0.1
    return dout, dlse


def run(state: dict):
    kind = state['kind']
    if kind in ('layer', 'teacher'):
        return state['student'](state['q'], state['k'], state['v'], 0)
    if kind == 'dense':
        return kernels.dense_attention(state['q'], state['k'], state['v'], state['used'], return_lse=True)
    layout = state['layout']
    if kind == 'sparse':
        return kernels.block_sparse_attention_lists(state['q'], state['k'], state['v'], state['lists'], layout)
    if kind == 'train':
        ins = (state['q'], state['k'], state['v'])
        if state['dlse'] is None:
            out = kernels.block_sparse_attention(*ins, state['mask'], layout)
            return (out.detach(), *torch.autograd.grad(out, ins, state['dout']))
        out, lse = kernels.block_sparse_attention(*ins, state['mask'], layout, return_lse=True)
        grads = torch.autograd.grad((out, lse), ins, (state['dout'], state['dlse']))
        return (out.detach(), lse.detach(), *grads)
    tiles, feats = kernels.gather_and_pool(state['x'], layout, None)
    kernels.scatter_tiles_(state['back'], tiles, layout, None)
    return tiles, feats, state['back']


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch


def _tiles(case: dict, shape: str) -> tuple[torch.Tensor, int, int]:
    """(rows [n, 128] of the packed sequence, -1 past a tile's real rows;
    reference tiles; video tiles). A span's tiles go h-block, w-block,
    t-block outer to inner, a tile's rows t, h, w; then the rows of no span."""
    used = _used(case)
    parts, covered = [], np.zeros(used, bool)
    spans = _spans(case)
    n_ref = 0
    for i, (start, (T, H, W)) in enumerate(spans):
        if i + 1 < len(spans):
            boxes = [(2 ** a, 2 ** b, 2 ** (7 - a - b)) for a in range(8) for b in range(8 - a)]
            fit = [s for s in boxes if s[0] <= T and s[1] <= H and s[2] <= W] or boxes
            st, sh, sw = min(fit, key=lambda s: (-(-T // s[0]) * -(-H // s[1]) * -(-W // s[2]),
                                                 max(s) / min(s), s))
        else:
            st, sh, sw = _grid(shape)
        ids = start + np.arange(T * H * W).reshape(T, H, W)
        covered[start:start + T * H * W] = True
        for hb in range(0, H, sh):
            for wb in range(0, W, sw):
                for tb in range(0, T, st):
                    rows = ids[tb:tb + st, hb:hb + sh, wb:wb + sw].reshape(-1)
                    parts.append(np.pad(rows, (0, TILE - rows.size), constant_values=-1))
        if i + 1 < len(spans):
            n_ref = len(parts)
    n_video = len(parts)
    rest = np.flatnonzero(~covered)
    for i in range(0, rest.size, TILE):
        rows = rest[i:i + TILE]
        parts.append(np.pad(rows, (0, TILE - rows.size), constant_values=-1))
    return torch.from_numpy(np.stack(parts)).cuda(), n_ref, n_video


def _select(case: dict, scores: torch.Tensor, n_ref: int, n_video: int, n: int) -> torch.Tensor:
    """[H, n, n] bool: per query tile and column block the highest scores, the
    diagonal forced, budgets rounded so that their mean is exact."""
    t, h, w = _grid(case['grid'])
    blocks = [(n_ref, n_video, t * h * w, _get(case, 'keep'))]
    if n_ref:
        rt, rh, rw = _grid(case['ref'])
        blocks.append((0, n_ref, rt * rh * rw, _get(case, 'ref_keep')))
    mask = torch.zeros(scores.shape[0], n, n, dtype=torch.bool, device='cuda')
    for lo, hi, tokens, ratio in blocks:
        cols = hi - lo
        if ratio >= 1.0:
            mask[:, :, lo:hi] = True
            continue
        s = scores[:, :n_video, lo:hi].clone()
        at = torch.arange(lo, hi, device='cuda')
        s[:, at, at - lo] = math.inf
        ideal = math.ceil(tokens / TILE)
        budget = ratio * ideal * ideal / cols
        if budget >= cols:
            k_lo, k_hi, frac = cols, cols, 0.0
        else:
            k_lo = min(max(1, math.floor(budget)), cols)
            k_hi, frac = min(k_lo + 1, cols), round(min(max(budget - k_lo, 0.0), 1.0), 12)
        ramp = np.floor(np.arange(n_video + 1, dtype=np.float64) * frac)
        allowed = k_lo + torch.from_numpy(ramp[1:] > ramp[:-1]).cuda().long()
        top = torch.sort(s, dim=-1, descending=True, stable=True)[1][..., :k_hi]
        keep = (torch.arange(k_hi, device='cuda') < allowed[:, None]).expand(top.shape)
        mask[:, :n_video].scatter_(2, top + lo, keep)
    mask[:, n_video:] = True
    mask[:, :, n_video:] = True
    return mask


def _to_tiles(x: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
    """One head [S, D] -> [n, 128, D] in 64 bits, 0 past the real rows."""
    return torch.where(rows[..., None] >= 0, x[rows.clamp(min=0)].double(), 0.0)


def _attend(q, k, v, mask, count, virtual=None, dout=None, dlse=None):
    """One head: q, k, v [n, 128, D], mask [n, n], count [n] real rows.
    Returns out and lse, and dq, dk, dv for an output gradient. virtual: the
    dropped tiles stand for one key each, their mean, weighted by count."""
    scale = 1.0 / math.sqrt(D)
    out, lse = torch.empty_like(q), q.new_empty(q.shape[:2])
    grads = [torch.zeros_like(q) for _ in range(3)] if dout is not None else None
    slot = torch.arange(TILE, device='cuda')
    per_row = mask.sum(-1).tolist()
    order = torch.sort(mask.to(torch.uint8), dim=-1, descending=True, stable=True)[1]
    i = 0
    while i < len(per_row):
        j, most = i + 1, per_row[i]
        while j < len(per_row) and (j + 1 - i) * max(most, per_row[j]) <= 2048:
            most = max(most, per_row[j])
            j += 1
        idx = order[i:j, :most]
        kept = torch.arange(most, device='cuda') < mask[i:j].sum(-1)[:, None]
        ok = (kept[..., None] & (slot < count[idx][..., None])).reshape(j - i, 1, most * TILE)
        kk, vv = (x[idx].reshape(j - i, most * TILE, D) for x in (k, v))
        s = ((q[i:j] @ kk.transpose(1, 2)) * scale).masked_fill_(~ok, -math.inf)
        lse[i:j] = torch.logsumexp(s, -1)
        p = s.sub_(lse[i:j, :, None]).exp_()
        if most <= 256:
            o = p @ vv
        else:  # few rows, many keys: a product per key tile, added up
            per_tile = p.reshape(-1, TILE, most, TILE).transpose(1, 2).contiguous()
            o = (per_tile @ vv.reshape(-1, most, TILE, D)).sum(1)
        if virtual is not None:
            mean, total = virtual
            pv = torch.exp(q[i:j] @ mean.T * scale - lse[i:j, :, None]) * ~mask[i:j, None]
            o = (o + pv @ total) / (1.0 + pv @ count.double())[..., None]
        out[i:j] = o
        if dout is not None:
            do = dout[i:j]
            dsum = (do * o).sum(-1)
            if dlse is not None:
                dsum = dsum - dlse[i:j]
            ds = p * ((do @ vv.transpose(1, 2)) - dsum[..., None]) * scale
            grads[0][i:j] = ds @ kk
            grads[1].index_add_(0, idx.reshape(-1), (ds.transpose(1, 2) @ q[i:j]).reshape(-1, TILE, D))
            grads[2].index_add_(0, idx.reshape(-1), (p.transpose(1, 2) @ do).reshape(-1, TILE, D))
        i = j
    return out, lse, grads


def _dense(q, k, v):
    """One head [n, D]: out and lse, a slab of rows at a time."""
    out, lse = torch.empty_like(q), q.new_empty(q.shape[0])
    for i in range(0, q.shape[0], 4096):
        s = (q[i:i + 4096] @ k.T) / math.sqrt(D)
        lse[i:i + 4096] = torch.logsumexp(s, -1)
        out[i:i + 4096] = s.sub_(lse[i:i + 4096, None]).exp_() @ v
    return out, lse


def _pool(x, count, second=False):
    """[n, 128, D] -> [n, 3 D] mean, max, min, or (E[x^2], Var x)."""
    real = (torch.arange(TILE, device='cuda') < count[:, None])[..., None]
    c = count.clamp(min=1).double()[:, None]
    mean = x.sum(1) / c
    if second:
        dev = torch.where(real, x - mean[:, None], 0.0)
        return (x * x).sum(1) / c, (dev * dev).sum(1) / c
    return torch.cat([mean, x.masked_fill(~real, -math.inf).amax(1), x.masked_fill(~real, math.inf).amin(1)], -1)


def _logits(case, q, k, count, w, head):
    def dense(name):
        values, scale = w[name]
        x = values[head].float()
        return (x if scale is None else (x * scale[head])).to(torch.bfloat16).double()

    def embed(x, name):
        f = _pool(x, count)
        return f @ dense(name) + f[:, :D]

    out = embed(q, 'proj_q') @ embed(k, 'proj_k').T / math.sqrt(D)
    if _get(case, 'count'):
        out = out + _gain(case)[head].double() * torch.log(count.clamp(min=1).double())
    if _get(case, 'rank'):
        raw, _ = _pool(q, count, second=True)
        _, var = _pool(k, count, second=True)
        out = out + (raw @ dense('so_q')) @ (var @ dense('so_k')).T
    return out


def _heat(q, k, count, n_video):
    """[n_video, n] softmax mass of every (query tile, key tile) over all real keys."""
    n = q.shape[0]
    real = (torch.arange(TILE, device='cuda') < count[:, None]).reshape(-1)
    heat = q.new_empty(n_video, n)
    keys = k.reshape(-1, D)
    for i in range(0, n_video, 32):
        rows = q[i:min(i + 32, n_video)]
        s = ((rows.reshape(-1, D) @ keys.T) / math.sqrt(D)).masked_fill_(~real, -math.inf)
        p = s.sub_(torch.logsumexp(s, -1, keepdim=True)).exp_().reshape(-1, TILE, n, TILE).sum(-1)
        ok = torch.arange(TILE, device='cuda') < count[i:i + rows.shape[0], None]
        heat[i:i + rows.shape[0]] = torch.where(ok[..., None], p, 0.0).sum(1)
    return heat


@torch.no_grad()
def exact(case: dict, seed: int):
    kind, heads, used = case['kind'], case['heads'], _used(case)
    g = _generator(case, seed)
    q, k, v = _qkv(case, g)
    if kind == 'dense':
        out = torch.zeros(q.shape, dtype=torch.float64, device='cuda')
        lse = torch.zeros(q.shape[:2], dtype=torch.float64, device='cuda')
        for h in range(heads):
            out[:used, h], lse[:used, h] = _dense(*(x[:used, h].double() for x in (q, k, v)))
        return out, lse
    shapes = _get(case, 'shapes').split(',')
    layouts = [_tiles(case, s) for s in shapes]
    if kind in ('layer', 'teacher'):
        w = _weights(case, g) if kind == 'layer' else None
        out = torch.zeros(q.shape, dtype=torch.float64, device='cuda')
        for h, which in enumerate(_shape_of_head(case)):
            rows, n_ref, n_video = layouts[which]
            count = (rows >= 0).sum(-1)
            qt, kt, vt = (_to_tiles(x[:, h], rows) for x in (q, k, v))
            scores = _logits(case, qt, kt, count, w, h) if kind == 'layer' else _heat(qt, kt, count, n_video)
            mask = _select(case, scores[None], n_ref, n_video, rows.shape[0])[0]
            virtual = None
            if _get(case, 'comp'):
                virtual = (kt.sum(1) / count.clamp(min=1).double()[:, None], vt.sum(1))
            o = _attend(qt, kt, vt, mask, count, virtual)[0]
            out[rows[rows >= 0], h] = o[rows >= 0]
        return out
    rows, n_ref, n_video = layouts[0]
    n, count = rows.shape[0], (rows >= 0).sum(-1)
    if kind == 'permute':
        tiles = torch.stack([_to_tiles(k[:, h], rows).reshape(-1, D) for h in range(heads)], 1)
        feats = torch.stack([_pool(_to_tiles(k[:, h], rows), count) for h in range(heads)])
        back = torch.cat([k.double(), k.new_zeros(1, heads, D).double()])
        return tiles, feats, back
    mask = _select(case, _scores(case, n_video, g), n_ref, n_video, n)
    dout = dlse = None
    if kind == 'train':
        dout, dlse = _out_grads(case, n, g)
        dout = (dout * (rows >= 0).reshape(-1, 1, 1)).double()
    outs = [torch.empty(n * TILE, heads, D, dtype=torch.float64, device='cuda') for _ in range(4 if dout is not None else 1)]
    lses = torch.empty(heads, n * TILE, dtype=torch.float64, device='cuda')
    for h in range(heads):
        qt, kt, vt = (_to_tiles(x[:, h], rows) for x in (q, k, v))
        o, l, grads = _attend(qt, kt, vt, mask[h], count,
                              dout=None if dout is None else dout[:, h].reshape(n, TILE, D),
                              dlse=None if dlse is None else dlse[h].double().reshape(n, TILE))
        lses[h] = l.reshape(-1)
        for to, x in zip(outs, [o] + (grads or [])):
            to[:, h] = x.reshape(-1, D)
    if kind == 'sparse':
        return outs[0]
    return (outs[0], lses, *outs[1:]) if dlse is not None else tuple(outs)
