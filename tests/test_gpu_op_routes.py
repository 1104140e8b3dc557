"""Calls of the ops that the dispatcher has to see still reach it (tracing,
fake tensors, gradients, transforms, function modes), ordinary calls give the
same result as the registered op, and in-place ops raise their argument's
version on both ways."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from miowtion_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu


def _args():
    lay = helpers.product_layout(*helpers.small_layout(), device='cuda')
    x = torch.randn(lay.seq_len, 4, 128, device='cuda').to(torch.bfloat16)
    return lay, (x, lay.gather_index, lay.slot_valid, lay.valid_count, torch.arange(4, device='cuda'),
                 True, True, False)


def test_ordinary_call_matches_the_registered_op():
    _, args = _args()
    for a, b in zip(ops.gather(*args), torch.ops.veda.gather(*args)):
        assert torch.equal(a, b)
    with torch.no_grad():
        x = args[0].clone().requires_grad_()
        assert not ops.gather(x, *args[1:])[0].requires_grad


def test_traced_calls_record_the_op():
    _, args = _args()
    graph = make_fx(lambda x: ops.gather(x, *args[1:])[1])(args[0])
    assert any(n.target is torch.ops.veda.gather.default for n in graph.graph.nodes)


def test_fake_tensors_take_the_fake_kernel():
    _, args = _args()
    with FakeTensorMode() as mode:
        fake = [mode.from_tensor(a) if isinstance(a, torch.Tensor) else a for a in args]
        out = ops.gather(*fake)
    assert tuple(out[0].shape) == (args[1].numel(), 4, 128)


def test_gradients_are_refused_as_by_the_op():
    _, args = _args()
    x = args[0].clone().requires_grad_()
    out = ops.gather(x, *args[1:])[1]
    assert out.requires_grad
    with pytest.raises(RuntimeError, match='autograd'):
        out.sum().backward()


def test_function_modes_see_the_op():
    class Mode(torch.overrides.TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Mode.seen += 'veda' in str(func)
            return func(*args, **(kwargs or {}))

    _, args = _args()
    with Mode():
        via_op = torch.ops.veda.gather(*args)
        before = Mode.seen
        via_fn = ops.gather(*args)
    assert Mode.seen - before == before
    assert torch.equal(via_op[0], via_fn[0])


def test_in_place_ops_raise_the_version():
    lay, args = _args()
    tiles = ops.gather(*args)[0]
    for call in (ops.scatter_, torch.ops.veda.scatter_):
        out = torch.zeros(lay.seq_len + 1, 4, 128, dtype=torch.bfloat16, device='cuda')
        before = out._version
        call(out, tiles, lay.scatter_index, lay.slot_valid, args[4])
        assert out._version > before


@pytest.mark.parametrize('make,ordinary', [
    (lambda: torch.ones(3, device='cuda'), True),
    (lambda: torch.ones(6, device='cuda')[::2], True),
    (lambda: torch._neg_view(torch.ones(3, device='cuda')), False),
    (lambda: torch.ones(3, dtype=torch.complex64, device='cuda').conj().imag, False),
    (lambda: torch.ones(3, dtype=torch.complex64, device='cuda').conj(), False),
    (lambda: torch._efficientzerotensor(3, device='cuda'), False),  # its address is null
    (lambda: torch.ones(3, device='cuda').requires_grad_(), False),
])
def test_verdict_on_tensors_whose_memory_is_not_their_value(make, ordinary):
    assert ops._ordinary((make(),), ((torch.Tensor,),)) == ordinary
    assert not ops._ordinary((make(),), ((int,),))


def test_lazily_negated_tensors_arrive_with_their_values():
    lay, args = _args()
    for x in (torch._neg_view(args[0]), torch._neg_view(args[0][:, 1:])):
        heads = torch.arange(x.shape[1], device='cuda')
        for a, b in zip(ops.gather(x, *args[1:4], heads, *args[5:]),
                        torch.ops.veda.gather(x, *args[1:4], heads, *args[5:])):
            assert torch.equal(a, b)
        assert torch.equal(ops.gather(x, *args[1:4], heads, *args[5:])[0],
                           ops.gather(x.resolve_neg(), *args[1:4], heads, *args[5:])[0])
    z = torch.randn(lay.seq_len, 4, 2, device='cuda')
    lse = torch.view_as_complex(z).conj().imag
    assert lse.is_neg()
    call = (lay.gather_index, lay.slot_valid, args[4])
    assert torch.equal(ops.gather_lse(lse, *call), torch.ops.veda.gather_lse(lse, *call))
    assert torch.equal(ops.gather_lse(lse, *call), ops.gather_lse(-z[..., 1], *call))


def test_inference_mode_as_by_the_op():
    lay, args = _args()
    kept = torch.zeros(lay.seq_len + 1, 4, 128, dtype=torch.bfloat16, device='cuda')
    with torch.inference_mode():
        fresh = torch.zeros_like(kept)
        tiles = ops.gather(*args)[0]
        assert tiles.is_inference() and torch.ops.veda.gather(*args)[0].is_inference()
        for call in (ops.scatter_, torch.ops.veda.scatter_):
            before = kept._version
            call(kept, tiles, lay.scatter_index, lay.slot_valid, args[4])
            assert kept._version > before
            call(fresh, tiles, lay.scatter_index, lay.slot_valid, args[4])
    assert torch.equal(kept, fresh)
    assert not ops.gather(*args)[0].is_inference()


def test_compiled_calls_record_the_op():
    _, args = _args()
    seen = []

    def backend(graph, _):
        seen.extend(str(n.target) for n in graph.graph.nodes)
        return graph.forward

    fn = torch.compile(lambda x: ops.gather(x, *args[1:])[1], backend=backend, fullgraph=True)
    assert torch.equal(fn(args[0]), ops.gather(*args)[1])
    assert any('gather' in s for s in seen)


def test_profiles_name_the_op():
    _, args = _args()
    with torch.autograd.profiler.profile() as prof:
        ops.gather(*args)
    assert any('veda::gather' in e.name for e in prof.function_events)


def test_a_layers_own_calls_are_ordinary(monkeypatch):
    """Every op that a layer calls takes the direct way (its numbers and
    flags are of the schema's own types)."""
    from miowtion_amd import attention as pa, mask as pm, plan as pplan, predictor as pp, tiling as pt
    verdicts, plain = [], ops._ordinary
    monkeypatch.setattr(ops, '_ordinary', lambda a, k: verdicts.append(plain(a, k)) or verdicts[-1])
    grid, shape = (4, 16, 16), pt.TileShape.parse('2x8x8')
    for comp in (False, True):
        config = pa.VedaConfig(target_budget=pm.Budget(ratio=0.5), zero_order_compensation=comp)
        clip = pa.ClipTiling(pa.PackedLayout((pa.VideoSpan(0, grid),), 1024, 1024), config, 'cuda')
        plan = pplan.TilePlan('clip', grid, [shape], [[0] * 4])
        layer = pp.LayerPredictor.random(4, 128, device='cuda')
        q, k, v = (t.cuda() for t in helpers.qkv(1024))
        for student in (pa.SparseStudent(clip, plan, pp.TileScorePredictor([layer])),
                        pa.OracleStudent(clip, plan)):
            student(q, k, v, 0)
    assert len(verdicts) > 20 and all(verdicts)
