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
