"""The float64 backward over tiles of receivers against the float64 one-wave-per-receiver backward: tile
sizes up to the limit, work pieces that cut sender runs, padding edges, rows without edges, a hub, an edge
permutation.  ds sums within one edge (the same bits); dx and dy add the same terms in another order."""

import ctypes

import numpy as np
import pytest
import torch

import e3j_amd
from e3j_amd import _lib, ops
from e3j_amd.graph import TileSchedule, csr_row_ptr, sort_edges
from e3j_amd.ops import _Table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x_irreps,channels", [("0e+1o+2e+3o", 64), ("0e+1o+2e", 128), ("0e", 64)])
@pytest.mark.parametrize("kind,tile_rows,max_work", [("even", 1, 256), ("even", 4, 256), ("hub", 3, 7), ("sorted", -1, 64), ("ordered", 4, 64),
                                                     ("one", 2, 256)])
def test_tiled_equals_receiver_rows(x_irreps, channels, kind, tile_rows, max_work):
    n, e = (1, 9) if kind == "one" else (90, 1500)
    gen = torch.Generator(device="cuda").manual_seed(e + channels)
    y_irreps = "0e+1o+2e+3o"
    module = e3j_amd.Convolution((x_irreps, y_irreps), y_irreps if x_irreps != "0e+1o+2e" else "0e+1o+2e",
                                 graph_ordering="NONE", layout="TRAILING_CHANNELS", avg_num_neighbors=30.0)
    dims = (module.source[0].dim, module.source[1].dim, module.params.num_out, module.params.num_scalars)
    rand = lambda *shape: torch.randn(shape, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    x, y, s, dm = rand(n, dims[0], channels), rand(e, dims[1]), rand(e, dims[3], channels), rand(n, dims[2], channels)
    receiver = torch.randint(0, max(1, n - 20), (e,), device="cuda", generator=gen).int()
    if kind == "hub":
        receiver[: e // 2] = 5
    sender = torch.randint(0, n, (e,), device="cuda", generator=gen).int()
    sender[::13] = 2 ** 31 - 1
    perm = None
    if kind == "sorted":
        receiver = receiver.sort().values
        other, ptr = sender, csr_row_ptr(receiver, n)
    else:
        receiver[::17] = 2 ** 31 - 1     # sorted behind the rows
        perm, other, ptr = sort_edges(receiver, sender, n)
    table = _Table.get(module._packed_coef("float64"), np.float64)
    sig, classes, _ = table.signature(dims, channels, module.layout)
    lib = _lib.load()
    limit = int(lib.e3j_amd_tile_rows_f64(sig))
    assert sig >= 0 and limit >= 1 and 1 <= lib.e3j_amd_tile_rows_default_f64(sig) <= limit
    order = torch.randperm(n, device="cuda", generator=gen).int() if kind == "ordered" else None
    sch = TileSchedule(other, ptr, perm, order, n, limit if tile_rows < 0 else min(tile_rows, limit), max_work)
    p = _lib.ConvParams(num_nodes=n, num_edges=e, num_coef=table.num_coef, num_x=dims[0], num_y=dims[1],
                        num_out=dims[2], num_scalars=dims[3], channels=channels, layout=_lib.LAYOUT_TRAILING,
                        val_dtype=_lib.F64, coef_idx_bytes=table.idx_bytes, signature=sig, coef_scale=1.0,
                        coef_classes=ctypes.cast(classes, ctypes.c_void_p).value,
                        row_order=order.data_ptr() if order is not None else None)
    pairs = []
    for tiled in (False, True):
        grads = [torch.full_like(t, float("nan")) for t in (x, y, s)]
        args = [x.data_ptr(), y.data_ptr(), s.data_ptr(), dm.data_ptr(), other.data_ptr(), ptr.data_ptr(),
                perm.data_ptr() if perm is not None else None]
        out = [g.data_ptr() for g in grads] + [int(torch.cuda.current_stream().cuda_stream)]
        if tiled:
            _lib.check(lib.e3j_amd_convolution_bwd_tiled_f64(ctypes.byref(p), *args, ctypes.byref(sch.struct), *out))
        else:
            _lib.check(lib.e3j_amd_convolution_bwd_receiver(ctypes.byref(p), None, *args, *out))
        pairs.append(grads)
    assert all(torch.isfinite(g).all() for g in pairs[1])
    assert torch.equal(pairs[0][2], pairs[1][2])
    for a, b, terms in ((pairs[0][0], pairs[1][0], e), (pairs[0][1], pairs[1][1], 16)):
        # sums of at most `terms` values in another order: sqrt(terms) roundings of the largest result
        assert float((a - b).abs().max()) <= 4 * terms ** 0.5 * 1.2e-16 * max(1.0, float(a.abs().max()))
    bad = TileSchedule(other, ptr, perm, None, n, limit + 1)
    assert lib.e3j_amd_convolution_bwd_tiled_f64(ctypes.byref(p), *args, ctypes.byref(bad.struct), *out) \
        == _lib.INVALID_ARGUMENT
    p.val_dtype = _lib.F32
    assert lib.e3j_amd_convolution_bwd_tiled_f64(ctypes.byref(p), *args, ctypes.byref(sch.struct), *out) \
        == _lib.UNIMPLEMENTED


@pytest.mark.parametrize("x_irreps,out_irreps,channels,kept", [
    ("0e+1o+2e+3o", "0e+1o+2e+3o", 128, True), ("0e+1o+2e", "0e+1o+2e", 64, True), ("0e+1o+2e", "0e+1o+2e", 64, False),
    ("0e+1o+2e", "0e+1o+2e", 192, True)])
def test_operator_above_the_threshold(x_irreps, out_irreps, channels, kept, monkeypatch):
    """Through the operator, with a row order (paired for a handle), just above the size from which tiles run,
    against the same call without them; 192 channels: a table compiled at run time."""
    y_irreps = "0e+1o+2e" if channels == 192 else "0e+1o+2e+3o"
    module = e3j_amd.Convolution((x_irreps, y_irreps), out_irreps, graph_ordering="RECEIVER",
                                 layout="TRAILING_CHANNELS", avg_num_neighbors=30.0)
    num_x, num_y, num_s = module.source[0].dim, module.source[1].dim, module.params.num_scalars
    n, e = 400, (1 if kept else 3) * 2 ** 23 // (num_x * channels) + 64
    gen = torch.Generator(device="cuda").manual_seed(channels)
    rand = lambda *shape: torch.randn(shape, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    receiver = torch.randint(0, n - 9, (e,), device="cuda", generator=gen).sort().values.int()
    sender = ((receiver + torch.randint(1, 40, (e,), device="cuda", generator=gen)) % n).int()
    sender[::13] = 2 ** 31 - 1
    x, y, s = (t.requires_grad_(True) for t in (rand(n, num_x, channels), rand(e, num_y), rand(e, num_s, channels)))
    dm = rand(n, module.params.num_out, channels)
    graph = ops.prepare_graph(sender, receiver, n) if kept else None
    taken = []
    monkeypatch.setattr(ops, "_tile_rows", lambda *a, f=ops._tile_rows, **k: taken.append((k, f(*a, **k))) or taken[-1][1])
    results = []
    for tile_rows in (-1, 0):
        with e3j_amd.config.use(tile_rows=tile_rows, jit=channels == 192):
            out = module(x, y, s, sender, receiver, graph=graph)
            results.append((out.detach(), *torch.autograd.grad(out, (x, y, s), dm)))
    assert taken[0][0] == {"f64": True} and taken[0][1] >= 1 and taken[1][1] == 0
    (out, dx, dy, ds), (out0, dx0, dy0, ds0) = results
    assert torch.equal(out, out0) and torch.equal(ds, ds0)
    for a, b, terms in ((dx0, dx, e // n), (dy0, dy, 16)):
        # sums of about `terms` values in another order: sqrt(terms) roundings of the largest result
        assert float((a - b).abs().max()) <= 8 * terms ** 0.5 * 1.2e-16 * float(a.abs().max())
