"""Rows and pieces of long rows in one launch (`e3j_amd_convolution_fwd_whole`): the same bits as the
call over the rows followed by the call over the pieces, whatever the number of pieces."""

import ctypes

import numpy as np
import pytest
import torch

import e3j_amd
from e3j_amd import _lib
from e3j_amd.graph import RowSegments, csr_row_ptr
from e3j_amd.ops import _Table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degrees", [
    (5, 0, 7),                       # no piece at all
    (64, 65, 0),                     # exactly the cap, one position past it
    (1, 128, 129, 3),                # one and two pieces
    (2000, 1, 70, 0, 0, 0, 0, 0, 90),    # many pieces of one row, rows without edges behind it
])
def test_one_call_equals_two(degrees):
    n, e = len(degrees), sum(degrees)
    gen = torch.Generator(device="cuda").manual_seed(e)
    module = e3j_amd.Convolution(("0e+1o+2e", "0e+1o+2e+3o"), "0e+1o+2e", graph_ordering="RECEIVER",
                                 layout="TRAILING_CHANNELS", avg_num_neighbors=30.0)
    receiver = torch.repeat_interleave(torch.arange(n, device="cuda"), torch.tensor(degrees, device="cuda")).int()
    sender = torch.randint(0, n, (e,), device="cuda", generator=gen).int()
    sender[::11] = 2 ** 31 - 1       # padding senders
    dims = (module.source[0].dim, module.source[1].dim, module.params.num_out, module.params.num_scalars)
    x, y, s = (torch.randn(shape, device="cuda", generator=gen)
               for shape in ((n, dims[0], 64), (e, dims[1]), (e, dims[3], 64)))
    table = _Table.get(module._packed_coef("float32"), np.float32)
    sig, scale, _ = table.signature(dims, 64, module.layout)
    assert sig >= 0
    ptr = csr_row_ptr(receiver, n)
    seg = RowSegments(ptr, n, e, 64, 64)
    lib, outs = _lib.load(), []
    for whole in (False, True):
        p = _lib.ConvParams(num_nodes=n, num_edges=e, num_coef=table.num_coef, num_x=dims[0], num_y=dims[1],
                            num_out=dims[2], num_scalars=dims[3], channels=64, layout=_lib.LAYOUT_TRAILING,
                            val_dtype=_lib.F32, coef_idx_bytes=table.idx_bytes, signature=sig, coef_scale=scale,
                            row_cap=64, row_piece=64)
        out = torch.full((n, dims[2], 64), float("nan"), device="cuda")
        args = (None, x.data_ptr(), y.data_ptr(), s.data_ptr(), sender.data_ptr(), ptr.data_ptr(), None,
                out.data_ptr(), int(torch.cuda.current_stream().cuda_stream))
        if not whole:
            _lib.check(lib.e3j_amd_convolution_fwd(ctypes.byref(p), *args))
        p.segments, p.max_segments = seg.buffer.data_ptr(), seg.max_segments
        if whole:   # without scratch rows the one call is refused
            assert lib.e3j_amd_convolution_fwd_whole(ctypes.byref(p), *args) == _lib.INVALID_ARGUMENT
        partials = torch.full((max(1, seg.max_segments), dims[2], 64), float("nan"), device="cuda")
        p.partials = partials.data_ptr()
        _lib.check((lib.e3j_amd_convolution_fwd_whole if whole else lib.e3j_amd_convolution_fwd)(ctypes.byref(p), *args))
        outs.append(out)
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
