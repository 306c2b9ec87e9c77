"""The tiled backward without dx (`e3j_amd_convolution_bwd_tiled_edges`): taken where x needs no gradient, and
dy and ds are what the kernel with dx gives."""

import contextlib
import ctypes

import numpy as np
import pytest
import torch

import e3j_amd
from e3j_amd import _lib, native, ops
from e3j_amd.options import config

pytestmark = pytest.mark.gpu


class _Calls:
    """The library with the names of the backward entries that the Python operators call on record."""

    def __init__(self, lib):
        self._lib, self.names = lib, []

    def __getattr__(self, name):
        if "convolution_bwd" in name:
            self.names.append(name)
        return getattr(self._lib, name)


@contextlib.contextmanager
def _native_calls():
    """The names of the tiled backwards that native calls make, which go through a callback to the same entries."""
    module, lib, names, keep = native.load(), _lib.load(), [], []
    entries = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in native._BOUND}
    watched = dict(entries)
    for name in ("e3j_amd_convolution_bwd_tiled", "e3j_amd_convolution_bwd_tiled_edges"):
        kind = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * len(getattr(lib, name).argtypes))

        def through(*args, name=name, entry=kind(entries[name])):
            names.append(name)
            return entry(*args)

        keep.append(kind(through))
        watched[name] = ctypes.cast(keep[-1], ctypes.c_void_p).value
    number = ctypes.addressof(config.number)
    module.bind(watched, number)
    try:
        yield names
    finally:
        module.bind(entries, number)


def _operands(n, channels, degree, irreps="0e+1o+2e+3o", dtype=torch.float32, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = e3j_amd.Convolution((irreps, irreps), irreps, graph_ordering="RECEIVER")
    receiver = torch.arange(n, device="cuda", dtype=torch.int32).repeat_interleave(degree)
    e = receiver.numel()
    sender = torch.randint(0, n, (e,), device="cuda", generator=g, dtype=torch.int32)
    sender[::7] = e3j_amd.DUMMY_INDEX
    rows = lambda *shape: torch.randn(shape, device="cuda", generator=g, dtype=dtype)   # noqa: E731
    x, y = rows(n, m.source[0].dim, channels), rows(e, m.source[1].dim)
    return m, x, y, rows(e, m.params.num_scalars, channels), sender, receiver, rows(n, m.target.dim, channels)


@pytest.mark.parametrize("n,degree,irreps", [(1, 1, "0e+1o+2e+3o"), (7, 3, "0e+1o+2e+3o"), (203, 31, "0e+1o+2e+3o"),
                                             (203, 31, "0e+1o+2e")])
@pytest.mark.parametrize("channels", [64, 128])
def test_same_edge_gradients(monkeypatch, n, degree, irreps, channels):
    if irreps == "0e+1o+2e":   # (the compiled table of that size has harmonics to degree 3)
        m, x, y, s, sender, receiver, dm = _operands(n, channels, degree)
        m = e3j_amd.Convolution((irreps, "0e+1o+2e+3o"), irreps, graph_ordering="RECEIVER")
        x, s, dm = x[:, :9].contiguous(), s[:, :m.params.num_scalars].contiguous(), dm[:, :m.target.dim].contiguous()
    else:
        m, x, y, s, sender, receiver, dm = _operands(n, channels, degree, irreps)
    native.load()   # (binds the entries it calls: not a call of them)
    lib = _Calls(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: lib)
    graph = ops.prepare_graph(sender, receiver, n)

    def edges(handle, x, wanted):
        yy, ss = y.clone().requires_grad_(True), s.clone().requires_grad_(True)
        out = m(x, yy, ss, sender, receiver, graph=handle)
        return torch.autograd.grad(out, {"ys": (yy, ss), "s": (ss,), "xys": (x, yy, ss)}[wanted], dm)

    leaf = x.clone().requires_grad_(True)
    _, dy, ds = edges(None, leaf, "xys")
    assert lib.names == ["e3j_amd_convolution_bwd_tiled"]
    lib.names.clear()
    # The same products and sums.  Which products the compiler fuses with their sum is its choice in each of the two
    # kernels, and the order in which the up to six waves of an edge add their parts of dy is not fixed: a rounding
    # of 2^-24 of a partial sum for each of at most 64 terms of a path in a row of dy or ds, partial sums that lie
    # within the largest value of all edges.
    def near(got, want):
        return float((got - want).abs().max()) <= 64 * 2.0 ** -24 * float(want.abs().max())

    def passes(handles):
        for handle in handles:
            for operand, wanted in ((x, "ys"), (leaf, "ys"), (x, "s")):   # (x a leaf that nobody asks about, too)
                got = edges(handle, operand, wanted)
                assert near(got[-1], ds)
                if wanted == "ys":
                    assert near(got[0], dy)
                    assert not got[0][sender >= n].any()
                assert not got[-1][sender >= n].any()

    form = "e3j_amd_convolution_bwd_tiled_edges"
    with _native_calls() as names:
        lib.names.clear()   # (asked for entries, not called)
        passes((None, graph, None, graph))
    # (the first backward of a handle makes its schedule, in Python)
    assert lib.names == [form] and names == [form] * 11
    lib.names.clear()
    monkeypatch.setattr(native, "call", lambda *a: None)   # (the Python operators)
    passes((None, graph))
    # (a node in Python knows which operands want gradients, not which of them are asked for)
    assert lib.names == [form, "e3j_amd_convolution_bwd_tiled", form] * 2


def test_dx_is_there_when_it_is_asked_for():
    """Beside a call without it, under create_graph, and where the kernels have no form without dx."""
    m, x, y, s, sender, receiver, dm = _operands(40, 64, 9)
    for _ in range(3):
        leaf, ss = x.clone().requires_grad_(True), s.clone().requires_grad_(True)
        out = m(leaf, y, ss, sender, receiver)
        (alone,) = torch.autograd.grad(out, leaf, dm, retain_graph=True)
        (ds,) = torch.autograd.grad(out, ss, dm, retain_graph=True, create_graph=True)
        (second,) = torch.autograd.grad((ds * s).sum(), leaf, retain_graph=True)
        out.backward(dm)
        # <dm, conv(x, y, s)> is linear in s: the gradient of <ds, s> with respect to x is dx
        bound = 3e-6 * float(leaf.grad.abs().max())
        assert float((alone - leaf.grad).abs().max()) <= bound and float((second - leaf.grad).abs().max()) <= 4 * bound
    for dtype, deterministic in ((torch.float64, False), (torch.float32, True)):
        m, x, y, s, sender, receiver, dm = _operands(40, 64, 9, dtype=dtype)
        with e3j_amd.config.use(deterministic=deterministic):
            for _ in range(3):
                ss = s.clone().requires_grad_(True)
                (got,) = torch.autograd.grad(m(x, y, ss, sender, receiver), ss, dm)
                leaf = x.clone().requires_grad_(True)
                want = torch.autograd.grad(m(leaf, y, ss, sender, receiver), (ss, leaf), dm)[0]
                eps = 1e-14 if dtype == torch.float64 else 3e-6
                assert float((got - want).abs().max()) <= eps * float(want.abs().max())


def test_the_entry_with_dx_still_needs_it():
    lib = _lib.load()
    m, x, y, s, sender, receiver, dm = _operands(8, 64, 4)
    table = ops._Table.get(m._packed_coef("float32"), np.float32)
    dims = (x.shape[1], y.shape[1], m.params.num_out, s.shape[1])
    sig, scale, flip = table.signature(dims, 64, m.layout)
    graph = ops.prepare_graph(sender, receiver, 8)
    other, row_ptr, perm, order = graph
    schedule = graph.schedule(int(lib.e3j_amd_tile_rows_default(sig)))
    p = _lib.ConvParams(num_nodes=8, num_edges=32, num_coef=table.num_coef, num_x=dims[0], num_y=dims[1], num_out=dims[2],
                        num_scalars=dims[3], channels=64, layout=m.layout.value, val_dtype=_lib.F32,
                        coef_idx_bytes=table.idx_bytes, signature=sig, coef_scale=scale, y_flip=flip,
                        row_order=order.data_ptr() if order is not None else None)
    args = [ctypes.byref(p), *(t.data_ptr() for t in (x, y, s, dm, other, row_ptr)),
            perm.data_ptr() if perm is not None else None, ctypes.byref(schedule.struct)]
    dy, ds = torch.empty_like(y), torch.empty_like(s)
    stream = int(torch.cuda.current_stream().cuda_stream)
    assert lib.e3j_amd_convolution_bwd_tiled(*args, None, dy.data_ptr(), ds.data_ptr(), stream) != 0
    assert lib.e3j_amd_convolution_bwd_tiled_edges(*args, None, ds.data_ptr(), stream) != 0
    assert lib.e3j_amd_convolution_bwd_tiled_edges(*args, dy.data_ptr(), None, stream) != 0
    assert lib.e3j_amd_convolution_bwd_tiled_edges(*args, dy.data_ptr(), ds.data_ptr(), stream) == 0
    torch.cuda.synchronize()
