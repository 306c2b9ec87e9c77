"""The convolution operator's common call in native code (`csrc/host/operators.cpp`).

`call` takes a module's call where its route is the plain one and answers None where it is not: the
Python operators of `ops.py` then run it (float16/32/64 tensors with an unrolled kernel, RECEIVER or NONE
ordering, the default kind of settings, no transform, mode or tracer at work).  Both give the same results
by the same library calls; this side spares a small graph's pass most of its host time.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import warnings

import torch

from . import _lib, ops
from .graph import MAX_WORK_EDGES, MIN_ROW_CAP, PARTIALS_BUDGET, ROW_PIECE
from .options import Config, GraphOrdering, Layout, config

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "_operators.so")

_BOUND = ("e3j_amd_prepare_rows", "e3j_amd_prepare_rows_workspace_bytes", "e3j_amd_row_segments_max",
          "e3j_amd_row_partials_bytes", "e3j_amd_convolution_fwd", "e3j_amd_convolution_fwd_whole",
          "e3j_amd_convolution_bwd_receiver", "e3j_amd_convolution_bwd_tiled",
          "e3j_amd_convolution_bwd_tiled_edges", "e3j_amd_convolution_bwd_tiled_f64",
          "e3j_amd_tile_schedule_num_work", "e3j_amd_tile_schedule_workspace_bytes", "e3j_amd_tile_schedule_build")
_module = None


def load():
    """The native module, bound to the kernel library this process has loaded; raises if it was not built."""
    global _module
    if _module is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(f"{LIB_PATH} is missing: build it with `python -m e3j_amd.build`")
        loader = importlib.machinery.ExtensionFileLoader("_operators", LIB_PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_operators", loader))
        loader.exec_module(module)
        lib = _lib.load()
        module.bind({name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _BOUND},
                    ctypes.addressof(config.number))
        _module = module
    return _module


_missing = False


def available():
    """`load()`'s module; None, said once, where this tree holds none that loads (not built, or built against another
    torch): the Python operators then make every call, by the same kernels."""
    global _missing
    if _module is None and not _missing:
        try:
            load()
        except ImportError as e:
            _missing = True
            warnings.warn(f"e3j_amd: calls of small graphs are slower without the native host side ({e})",
                          RuntimeWarning, stacklevel=2)
    return _module


#: no size reaches this: a route that is never taken
_NEVER = 1 << 62


def _plan(module, x: torch.Tensor, cfg: Config):
    """A plan for calls of `module` on tensors like `x`, False where such calls are not the plain ones."""
    ordering, layout = module.graph_ordering, module.layout
    if (x.device.type != "cuda" or x.dtype not in ops._VAL_DTYPES or ordering == GraphOrdering.SENDER
            or cfg.graph_cache or cfg.deterministic or not cfg.fixed_order_rows or cfg.debug_level
            or cfg.pair_rows is True
            or not all(-1 << 31 <= int(v) < 1 << 31 for v in (cfg.row_cap, cfg.locality_rounds, cfg.tile_rows))):
        return False
    code, val_np = ops._VAL_DTYPES[x.dtype]
    coef, params = module._packed_coef(val_np.__name__), module.params
    table = ops._Table.get(coef, val_np)
    trailing = layout == Layout.TRAILING_CHANNELS
    num_x, channels = (x.shape[1], x.shape[2]) if trailing else (x.shape[2], x.shape[1])
    dims = (int(num_x), int(module.source[1].dim), int(params.num_out), int(params.num_scalars))
    sig, scale, flip = table.signature(dims, int(channels), layout)
    if sig < 0 or available() is None:
        return False
    f64 = x.dtype == torch.float64
    p = _lib.ConvParams(
        num_coef=table.num_coef, num_x=dims[0], num_y=dims[1], num_out=dims[2], num_scalars=dims[3],
        channels=int(channels), layout=layout.value, val_dtype=code, coef_idx_bytes=table.idx_bytes, signature=sig,
        coef_scale=1.0 if f64 else scale, y_flip=flip, table_plan_state=_lib.PLAN_BUILD)
    if f64:
        p.coef_classes = ctypes.cast(scale, ctypes.c_void_p).value
    # the backward over tiles: always (float32), from a number of dx values on (float64), never
    tile_rows, values, values_kept = 0, _NEVER, _NEVER
    if trailing and x.dtype == torch.float32:
        tile_rows, values, values_kept = ops._tile_rows(sig), 0, 0
    elif f64:
        tile_rows = ops._tile_rows(sig, f64=True)
        values, values_kept = (ops.tile_values_f64(dims[0], dims[3], kept) or _NEVER for kept in (False, True))

    def fallback(x, y, s, dm, sender, receiver, graph, need_dx):
        meta = ops._make_meta(coef, x, y, s, params, ordering, None, layout)
        return ops._backward(x, y, s, dm, sender, receiver, meta, graph, need_dx)

    def make_graph(other, row_ptr, perm, order, num_nodes, segments, row_cap, row_piece):
        graph = ops.PreparedGraph(other, row_ptr, perm, order, num_nodes, ordering)
        if segments is not None:
            graph.adopt_segments(segments, row_cap, row_piece)
        return graph

    return load().Plan(
        bytes(p), table.device(x.device), code,
        dict(sorted=ordering != GraphOrdering.NONE, rounds=int(cfg.locality_rounds),
             unordered_rows=ops.UNORDERED_ROWS if int(cfg.locality_rounds) == Config.locality_rounds else 0,
             share_rows=trailing and x.dtype == torch.float32, row_cap=int(cfg.row_cap), min_row_cap=MIN_ROW_CAP,
             piece=ROW_PIECE, partials_budget=PARTIALS_BUDGET, tile_rows=tile_rows, max_work_edges=MAX_WORK_EDGES,
             tile_values=values, tile_values_kept=values_kept),
        fallback, make_graph, scale if f64 else None)


def call(module, x, y, s, sender, receiver, graph):
    """`module`'s convolution of the operands, or None."""
    cfg, number = config.state
    plans = module._plans   # the settings seen last and their plans
    if plans is None or plans[0] is not cfg:
        if module._plan_sets is None:
            module._plan_sets = {}
        sets = module._plan_sets
        if len(sets) >= 8 and cfg not in sets:
            sets.clear()
        plans = module._plans = (cfg, sets.setdefault(cfg, {}))
    try:
        key = (x.dtype, x.device, x.shape[1:], module.layout, module.graph_ordering)
        plan = plans[1].get(key)
    except (AttributeError, TypeError):   # not tensors: the operator says so
        return None
    if plan is None:
        if type(x) is not torch.Tensor and type(x) is not torch.nn.Parameter or x.ndim != 3 or not x.is_cuda:
            return None
        # the first call of a kind runs the Python operators, which say what may be wrong with it; the second
        # finds it here and makes the plan
        plans[1][key] = True
        return None
    if plan is True:
        plan = _plan(module, x, cfg)
        if config.state[1] != number:   # (another thread changed the settings under it: the plan may be of both)
            return None
        plans[1][key] = plan
    if plan is False:
        return None
    if graph is None:
        return _module.call(plan, x, y, s, sender, receiver, None, None, None, number)
    if not isinstance(graph, ops.PreparedGraph) or graph.ordering != module.graph_ordering or not graph.kept:
        return None
    adjacency = graph.native(plan, module, x, cfg)
    if adjacency is None:
        return None
    schedule = graph._schedules.get(plan.tile_rows) if plan.tile_rows else None
    graph.ready()
    return _module.call(plan, x, y, s, sender, receiver, adjacency, graph, schedule, number)
