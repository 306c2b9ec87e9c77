"""The float64 backward over tiles of receivers against the float64 one-wave-per-receiver backward: tile
sizes up to the limit, work pieces that cut sender runs, padding edges, rows without edges, a hub, an edge
permutation.  ds sums within one edge (the same bits); dx and dy add the same terms in another order."""

import ctypes

import numpy as np
import pytest
import torch

import e3j_amd
from e3j_amd import _lib
from e3j_amd.graph import TileSchedule, csr_row_ptr, sort_edges
from e3j_amd.ops import _Table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x_irreps,channels", [("0e+1o+2e+3o", 64), ("0e+1o+2e", 128), ("0e", 64)])
@pytest.mark.parametrize("kind,tile_rows,max_work", [("even", 1, 256), ("even", 4, 256), ("hub", 3, 7), ("sorted", -1, 64),
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
    sch = TileSchedule(other, ptr, perm, None, n, limit if tile_rows < 0 else min(tile_rows, limit), max_work)
    p = _lib.ConvParams(num_nodes=n, num_edges=e, num_coef=table.num_coef, num_x=dims[0], num_y=dims[1],
                        num_out=dims[2], num_scalars=dims[3], channels=channels, layout=_lib.LAYOUT_TRAILING,
                        val_dtype=_lib.F64, coef_idx_bytes=table.idx_bytes, signature=sig, coef_scale=1.0,
                        coef_classes=ctypes.cast(classes, ctypes.c_void_p).value)
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
