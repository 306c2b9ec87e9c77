"""Which way an operator call takes, with the library stubbed: no GPU needed."""

import types

import pytest
import torch
from torch.autograd import forward_ad

from e3j_amd import ops


def _blank(*like):
    """Results as the library gives them: written through pointers, unknown to autograd."""
    return tuple(torch.zeros(t.shape) for t in like)


def _operands():
    return torch.randn(4, 3, 2), torch.randn(5, 3), torch.randn(5, 2, 2), torch.randn(4, 3, 2)


@pytest.mark.parametrize("need_dx", [True, False])
def test_a_backward_drops_no_forward_mode_tangent(monkeypatch, need_dx):
    monkeypatch.setattr(ops, "_raw_backward", lambda meta, x, y, s, *rest, need_dx=True: _blank(x, y, s))
    x, y, s, dm = _operands()
    with torch.no_grad(), forward_ad.dual_level():
        dual = forward_ad.make_dual(dm, torch.ones_like(dm))
        with pytest.raises(NotImplementedError, match="jvp"):
            ops._backward(x, y, s, dual, None, None, None, object(), need_dx)
        assert len(ops._backward(x, y, s, dm, None, None, None, object(), need_dx)) == 3


def test_a_second_derivative_drops_no_forward_mode_tangent(monkeypatch):
    x, y, s, dm = _operands()
    ctx = types.SimpleNamespace(saved_tensors=(x, y, s, dm), index=(None, None), meta=None, graph=object())
    monkeypatch.setattr(ops, "_raw_second", lambda meta, x, y, s, dm, *rest: _blank(x, y, s, dm))
    monkeypatch.setattr(ops, "_raw_forward", lambda *a: _blank(dm)[0])
    monkeypatch.setattr(ops, "_raw_backward", lambda *a: _blank(x, y, s))
    with torch.no_grad():
        assert len(ops._ConvolutionBwd.backward(ctx, x, y, s)) == 8
        with forward_ad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
            ops._ConvolutionBwd.backward(ctx, forward_ad.make_dual(x, torch.ones_like(x)), y, s)
