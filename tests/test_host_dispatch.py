"""Calls of the forward operators past their autograd formula: where it may be passed by and where not."""
import pytest
import torch

from savanna_amd import _lib
from savanna_amd.kernels.cgcg.interface import interleaved_source, planar_source


def _probe():
    """An operator call that reports whether the autograd keys are excluded around it."""
    seen = []
    return seen, lambda *a: seen.append(
        torch._C._dispatch_tls_local_exclude_set().has(torch._C.DispatchKey.AutogradFunctionality))


def test_formula_is_kept_while_gradients_are_recorded():
    seen, op = _probe()
    _lib._run(op)
    with torch.no_grad():
        _lib._run(op)
    _lib._run(op)
    assert seen == [False, True, False]


def test_formula_is_kept_under_function_transforms():
    seen, op = _probe()
    with torch.no_grad():
        torch.func.vmap(lambda t: (_lib._run(op), t)[1])(torch.ones(2))
    assert seen == [False]


@pytest.mark.parametrize("g,dg,L,bs", [(1, 1, 1, 1), (1, 1, 5, 2), (4, 1, 1, 2), (1, 16, 3, 1), (3, 8, 1, 2), (2, 16, 7, 2)])
def test_views_are_recognised_and_separate_tensors_are_not(g, dg, L, bs):
    feat = torch.randn(bs, L, g, dg, 3)
    C, B, x = feat.unbind(4)
    src = interleaved_source(x, B, C)
    assert src is not None and src.data_ptr() == feat.data_ptr() and torch.equal(src, feat)
    plan = torch.randn(bs, L, 3, g, dg)
    C, B, x = plan.unbind(2)
    src = planar_source(x, B, C)
    assert src is not None and src.data_ptr() == plan.data_ptr() and torch.equal(src, plan)
    x, B, C = (torch.randn(bs, L, g, dg) for _ in range(3))
    assert interleaved_source(x, B, C) is None and planar_source(x, B, C) is None
