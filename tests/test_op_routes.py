"""Which calls of an op go through the dispatcher: the verdicts that need no
GPU. (The routes' results are compared in test_gpu_op_routes.py.)"""

import subprocess
import sys

import torch

from miowtion_amd import ops

ROOT = __file__.rsplit('/', 2)[0]


REST = (None, True, True, False)  # gather's heads and flags


def test_symbolic_traces_record_the_op():
    graph = torch.fx.symbolic_trace(lambda x, i, ok, n: ops.gather(x, i, ok, n, *REST)).graph
    assert any('veda' in str(n.target) and 'gather' in str(n.target) for n in graph.nodes)


def test_an_object_with_torch_function_is_asked():
    class Duck:
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            return str(func)

    assert 'gather' in ops.gather(*[Duck()] * 4, *REST)


def test_arguments_of_another_type_are_left_to_the_op():
    kinds = ops.predictor_logits._kinds
    assert kinds[2] == (float,) and kinds[3] == (torch.Tensor, type(None))
    assert ops._ordinary((), kinds)
    for kind, ok, other in (((float,), 1.0, 1), ((int,), 1, True), ((bool,), True, 1),
                            ((torch.Tensor, type(None)), None, torch.nn.Parameter(torch.zeros(1)))):
        assert ops._ordinary((ok,), (kind,)) and not ops._ordinary((other,), (kind,))
    assert not ops._ordinary((None,) * 8, kinds)  # more than the op takes
    assert not ops._ordinary((torch.zeros(1),), kinds)  # not on the GPU


def test_profiled_calls_show_as_the_op():
    with torch.autograd.profiler.profile():
        assert not ops._ordinary((), ())
    assert ops._ordinary((), ())


def test_import_without_a_gpu_build_of_torch():
    code = ('import torch\n'
            "if hasattr(torch._C, '_cuda_getCurrentRawStream'): del torch._C._cuda_getCurrentRawStream\n"
            'torch.cuda._is_compiled = lambda: False\n'
            'from miowtion_amd import ops\n'
            'try: ops.gather(*[torch.zeros(1, 1, 128, dtype=torch.bfloat16)] * 5, True, True, False)\n'
            'except NotImplementedError: print("refused")\n')
    out = subprocess.run([sys.executable, '-c', code], cwd=ROOT, capture_output=True, text=True)
    assert out.stdout.strip() == 'refused', out.stderr
