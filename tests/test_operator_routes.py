"""Which way an operator call takes, with the library stubbed: no GPU needed."""

import pickle
import types
import warnings

import pytest
import torch
from torch.autograd import forward_ad

from e3j_amd import Convolution, native, ops
from e3j_amd.options import Config, config


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


def test_a_module_pickled_without_plans_runs():
    """As one was before modules kept plans of native calls; and plans do not travel with a module."""
    module = Convolution(("0e+1o", "0e+1o"), "0e+1o", graph_ordering="RECEIVER")
    state = {k: v for k, v in vars(module).items() if "plan" not in k}
    old = pickle.loads(pickle.dumps(module))
    vars(old).clear()
    vars(old).update(state)
    x, index = torch.zeros(2, 4, 8), torch.zeros(3, dtype=torch.int32)
    operands = x, torch.zeros(3, 4), torch.zeros(3, module.params.num_scalars, 8), index, index
    for m in (old, module):
        for _ in range(3):
            with pytest.raises(RuntimeError, match="GPU memory"):
                m(*operands)
    module._plan_sets, module._plans = {"settings": object}, ("settings", {})
    twin = pickle.loads(pickle.dumps(module))
    assert twin._plans is None and not twin._plan_sets and twin.params == module.params


@pytest.mark.parametrize("there", [False, True])
def test_a_tree_without_its_native_host_side_says_so_once(monkeypatch, tmp_path, there):
    """Not built, or not a module that loads here."""
    path = tmp_path / "_operators.so"
    if there:
        path.write_bytes(b"of another torch")
    for name, value in (("LIB_PATH", str(path)), ("_module", None), ("_missing", False)):
        monkeypatch.setattr(native, name, value)
    with pytest.warns(RuntimeWarning, match="native host side"):
        assert native.available() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert native.available() is None
    with pytest.raises(ImportError):
        native.load()


def test_a_plan_made_while_the_settings_change_is_not_kept(monkeypatch):
    module = Convolution(("0e+1o", "0e+1o"), "0e+1o", graph_ordering="RECEIVER")
    x = torch.zeros(2, 4, 64)
    key, cfg = (x.dtype, x.device, x.shape[1:], module.layout, module.graph_ordering), config()
    module._plan_sets = {cfg: {key: True}}   # (a call of this kind was made)

    def plan(*args):
        config(tile_rows=0)   # another thread's
        return object()

    before = config.state
    monkeypatch.setattr(native, "_plan", plan)
    try:
        assert native.call(module, x, None, None, None, None, None) is None
    finally:
        config._enter(*before)
    assert module._plan_sets[cfg] == {key: True}


@pytest.mark.parametrize("setting", [dict(row_cap=10 ** 10), dict(locality_rounds=2 ** 31)])
def test_settings_past_32_bits_are_left_to_the_python_operators(setting):
    module = Convolution(("0e+1o+2e+3o", "0e+1o+2e+3o"), "0e+1o+2e+3o", graph_ordering="RECEIVER")
    x = types.SimpleNamespace(dtype=torch.float32, device=torch.device("cuda", 0), shape=torch.Size((2, 16, 64)))
    assert native._plan(module, x, Config(**setting)) is False
