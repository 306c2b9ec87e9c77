"""The second-order backward (`e3j_amd_convolution_bwd_bwd`) through autograd, against the float64 oracle:
each gradient is a sum of two or three first-order results, so the reference and the magnitude of its
terms are sums of the oracle's (the rounding allowance of `helpers.assert_parity` applies to the sum)."""

import ctypes

import numpy as np
import pytest
import torch

from e3j_amd import _lib, config, ops
from e3j_amd.codegen.gen_conv import BUILTIN_SIGNATURES
from e3j_amd.convolution import Convolution
from tests import helpers as H

pytestmark = pytest.mark.gpu

DUMMY = int(np.iinfo(np.int32).max)


def _graph(rng, kind):
    """Receivers sorted (except "shuffled"); sizes at the edges of tiles, of batches of 64 positions and of
    the pieces of long rows."""
    if kind == "single":                       # one edge, one node
        return 1, np.zeros(1, np.int32), np.zeros(1, np.int32)
    if kind == "hub":                          # one row of 300 positions, past row_cap, pieces and work items
        n = 37
        degree = rng.integers(0, 9, size=n)    # some rows are empty
        degree[5] = 300
    elif kind == "many":                       # past the rows that keep their index order; a hub, empty rows
        n = 300
        degree = rng.integers(0, 4, size=n)
        degree[7] = 200
    else:                                      # rows of 63, 64, 65 positions; padding edges; the last tile is short
        n = 13
        degree = np.array([63, 64, 65, 0, 1, 2, 7, 8, 9, 0, 30, 31, 4])
    rcv = np.repeat(np.arange(n), degree).astype(np.int32)
    snd = rng.integers(0, n, size=rcv.shape[0]).astype(np.int32)
    if kind == "padding":
        snd[rng.random(snd.shape[0]) < 0.2] = DUMMY
        snd[:64] = DUMMY                       # a whole batch without a live position
    if kind == "shuffled":
        order = rng.permutation(rcv.shape[0])
        snd, rcv = snd[order], rcv[order]
    return n, snd, rcv


#: (256 channels: other tiles, the same edge loops as at 128; two graphs keep the oracle quick)
CASES = [(sig, kind) for sig in BUILTIN_SIGNATURES if sig[4] >= 64
         for kind in (("single", "hub") if sig[4] == 256 else ("single", "hub", "padding", "shuffled"))]


def _compare_with_oracle(sig, kind, monkeypatch, handle=False, ordered=False):
    """Second derivatives through autograd, which must come from one call of the library.  `handle`: the
    adjacency from `prepare_graph`; `ordered`: the rows then have an order."""
    name, xi, yi, oi, channels = sig
    rng = np.random.default_rng(channels + len(kind))
    module = Convolution((xi, yi), oi, graph_ordering="NONE" if kind == "shuffled" else "RECEIVER")
    n, snd, rcv = _graph(rng, kind)
    num_x, num_y, num_z, num_s = (module.source[0].dim, module.source[1].dim, module.target.dim,
                                  module.params.num_scalars)
    x, y, s, dm = H.random_operands(rng, n, len(snd), num_x, num_y, num_s, channels, num_z)
    x2, y2, s2, _ = H.random_operands(rng, n, len(snd), num_x, num_y, num_s, channels, num_z)
    pad = snd == DUMMY
    dev = {k: torch.from_numpy(v.copy()).cuda() for k, v in dict(x=x, y=y, s=s, dm=dm, x2=x2, y2=y2, s2=s2).items()}
    for k in ("y", "s", "y2", "s2"):           # padding edges hold anything
        dev[k][torch.from_numpy(pad)] = float("nan")
    results = []
    monkeypatch.setattr(ops, "_raw_second", lambda *a, f=ops._raw_second: results.append(f(*a)) or results[-1])
    leaves = [dev[k].requires_grad_(True) for k in ("x", "y", "s", "dm")]
    index = torch.from_numpy(snd).cuda(), torch.from_numpy(rcv).cuda()
    with config.use(locality_rounds=1):        # (graphs as small as most of these keep the index order at 2)
        graph = ops.prepare_graph(*index, n, module.graph_ordering) if handle else None
    orders = []
    monkeypatch.setattr(ops, "_fill_params",
                        lambda *a, f=ops._fill_params, **k: orders.append(k.get("row_order")) or f(*a, **k))
    out = module(*leaves[:3], *index, graph=graph)
    first = torch.autograd.grad(out, leaves[:3], leaves[3], create_graph=True)
    got = torch.autograd.grad(first, leaves, [dev["x2"], dev["y2"], dev["s2"]])
    assert len(results) == 1 and results[0] is not None     # (None: the first-order operators composed them)
    if ordered:                                # of forward, backward and second-order backward
        assert len(orders) == 3 and not any(torch.equal(o.cpu(), torch.arange(n).int()) for o in orders)
    live = ~pad
    idx = np.asarray(module.coef.idx, dtype=np.int64)
    val, mix = np.asarray(module.coef.val, dtype=np.float32), module._mix.mix_indices
    args = (idx[:, :3], val, mix)
    e = dict(snd=snd[live], rcv=rcv[live])
    y, s, y2, s2 = y[live], s[live], y2[live], s2[live]
    f = [H.forward_reference(*args, a, b, c, e["snd"], e["rcv"], num_z) for a, b, c in
         ((x2, y, s), (x, y2, s), (x, y, s2))]
    b = [H.backward_reference(*args, a, c, d, e["snd"], e["rcv"], dm) for a, c, d in
         ((x2, y, s), (x, y2, s), (x, y, s2))]
    g = [t.detach().cpu().numpy() for t in got]
    pick = lambda which, grad, part: sum(b[w][part][grad] for w in which)  # noqa: E731
    for name_, result, ref, mag in (
            ("x", g[0], pick((1, 2), 0, 0), pick((1, 2), 0, 1)),
            ("y", g[1][live], pick((0, 2), 1, 0), pick((0, 2), 1, 1)),
            ("s", g[2][live], pick((0, 1), 2, 0), pick((0, 1), 2, 1)),
            ("dm", g[3], sum(t[0] for t in f), sum(t[1] for t in f))):
        H.assert_parity(result, ref, mag, f"{name} {kind} gradient of {name_}")
    assert not g[1][pad].any() and not g[2][pad].any()


@pytest.mark.parametrize("sig,kind", CASES, ids=[f"{s[0]}-{k}" for s, k in CASES])
def test_second_order_matches_oracle(sig, kind, monkeypatch):
    _compare_with_oracle(sig, kind, monkeypatch)


@pytest.mark.parametrize("channels,variant", [(64, 1), (128, 4)])
def test_tiles_that_only_the_first_order_backward_can_hold(channels, variant, monkeypatch):
    """A first-order launch variant whose tiles take less LDS a row allows more rows than the second-order
    kernel holds: `config(tile_rows=...)` is cut to what each of them takes."""
    sig = next(s for s in BUILTIN_SIGNATURES if s[0] == f"l3_l3_to_l3_k{channels}")
    lib = _lib.load()
    lib.e3j_amd_set_launch_variant.argtypes = [ctypes.c_int32, ctypes.c_int32]
    lib.e3j_amd_set_launch_variant.restype = None
    lib.e3j_amd_set_launch_variant(0, variant)
    try:
        ids = [i for i in range(lib.e3j_amd_num_signatures())
               if lib.e3j_amd_signature_name(i).decode().startswith(sig[0]) and lib.e3j_amd_tile_rows_second(i) > 0]
        rows, least = lib.e3j_amd_tile_rows(ids[0]), lib.e3j_amd_tile_rows_second(ids[0])
        assert rows > least >= 1
        with config.use(tile_rows=rows):
            _compare_with_oracle(sig, "hub", monkeypatch)
    finally:
        lib.e3j_amd_set_launch_variant(0, 0)


ORDERED = [(f"{table}_k{k}", kind, handle) for table, k in (("l3_l3_to_l3", 64), ("l3_l3_to_l3", 128), ("l2_l3_to_l2", 64))
           for kind, handle in (("many", False), ("hub", True), ("padding", True), ("shuffled", True))]
ORDERED += [("l3_l3_to_l3_k256", "hub", True), ("l0_l3_to_l3_k64", "many", False)]


@pytest.mark.parametrize("name,kind,handle", ORDERED)
def test_rows_with_an_order(name, kind, handle, monkeypatch):
    """Rows and tiles in a locality order: prepared by the call (more rows than keep their index order) and by a
    handle, which pairs rows too."""
    sig = next(s for s in BUILTIN_SIGNATURES if s[0] == name)
    _compare_with_oracle(sig, kind, monkeypatch, handle, ordered=True)


@pytest.mark.parametrize("handle", [False, True])
def test_capture_and_replay(handle):
    """Forward, backward and second-order backward (and the preparation of sorted rows) recorded into a graph: every
    replay on rewritten operands equals the eager call."""
    n, snd, rcv = _graph(np.random.default_rng(5), "many")
    module = Convolution(("0e+1o+2e", "0e+1o+2e+3o"), "0e+1o+2e", graph_ordering="RECEIVER")
    dims = module.source[0].dim, module.source[1].dim, module.params.num_scalars, module.target.dim
    shapes = [(n, dims[0], 64), (len(snd), dims[1]), (len(snd), dims[2], 64), (n, dims[3], 64)]
    operands = [torch.zeros(shape, device="cuda") for shape in (*shapes, *shapes[:3])]    # x, y, s, dm and the cotangents
    x, y, s, dm = operands[:4]
    index = torch.from_numpy(snd).cuda(), torch.from_numpy(rcv).cuda()
    meta = ops._make_meta(module._packed_coef("float32"), x, y, s, module.params, module.graph_ordering, None, module.layout)
    kept = ops.prepare_graph(*index, n) if handle else None

    def passes():
        graph = kept or ops._prepare_graph(meta.ordering, n, *index, pieces=ops._row_pieces(meta, x, len(snd)))
        out = ops._raw_forward(meta, x, y, s, *index, graph)
        first = ops._raw_backward(meta, x, y, s, dm, *index, graph)
        return out, *first, *ops._raw_second(meta, *operands, *index, graph)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        passes()                                          # warm-up outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        recorded = passes()
    for trial in range(4):
        for t in operands:
            t.copy_(torch.randn_like(t))
        eager = passes()
        for t in recorded:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for which, (a, b) in enumerate(zip(recorded, eager)):
            if which in (0, 3, 6, 7):                     # out, ds, and the second-order ds and dm: fixed orders
                assert torch.equal(a, b), (trial, which)
            else:                                         # atomics: equal up to summation order
                assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max()), (trial, which)


def test_no_scratch_rows_without_the_fixed_order(monkeypatch):
    """`config(fixed_order_rows=False)` promises no scratch rows: the second derivatives are then composed from the
    first-order operators, which add the pieces of long rows with atomics."""
    n, snd, rcv = _graph(np.random.default_rng(3), "hub")
    module = Convolution(("0e+1o", "0e+1o+2e"), "0e+1o+2e", graph_ordering="RECEIVER")
    rand = lambda *shape: torch.randn(shape, device="cuda")  # noqa: E731
    dims = module.source[0].dim, module.source[1].dim, module.params.num_scalars, module.target.dim
    leaves = [t.requires_grad_(True) for t in (rand(n, dims[0], 64), rand(len(snd), dims[1]), rand(len(snd), dims[2], 64),
                                               rand(n, dims[3], 64))]
    second = [rand(*t.shape) for t in leaves[:3]]
    index = torch.from_numpy(snd).cuda(), torch.from_numpy(rcv).cuda()
    results = []
    for fixed in (False, True):
        graph = ops.prepare_graph(*index, n)
        with config.use(fixed_order_rows=fixed):
            out = module(*leaves[:3], *index, graph=graph)
            first = torch.autograd.grad(out, leaves[:3], leaves[3], create_graph=True)
            results.append(torch.autograd.grad(first, leaves, second))
        assert any(s._partials for s in graph._segments.values()) == fixed
    for a, b in zip(*results):
        # sums of at most 300 terms in another order, twice: sqrt(300) roundings of the largest value
        assert float((a - b).abs().max()) <= 2 * 300 ** 0.5 * 1.2e-7 * float(b.abs().max())


#: tables the library is not built for: shapes of 64 channels at 192, and fewer waves per SIMD for the larger
#: tables (`second_shapes`: two in both kernels; two and one)
RUN_TIME = [("0e+1o+2e", "0e+1o+2e", "0e+1o+2e", 64), ("0e+1o+2e", "0e+1o+2e", "0e+1o+2e", 192),
            ("0e+1o+2e", "0e+1o+2e+3o+4e", "0e+1o+2e+3o+4e", 64),
            ("0e+1o+2e+3o+4e", "0e+1o+2e+3o+4e", "0e+1o+2e", 128)]


@pytest.mark.parametrize("xi,yi,oi,channels", RUN_TIME)
def test_run_time_compiled_tables(xi, yi, oi, channels, monkeypatch):
    with config.use(jit=True):
        _compare_with_oracle(("run-time table", xi, yi, oi, channels), "hub", monkeypatch)
