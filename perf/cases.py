"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values; `listed()` names the ones that are followed over time and
`draw(rng)` gives further ones of the same ranges.  `prepare` makes what a user's program holds
before the call, `run` is one pass through the public entry points, `work` the bytes and operations
a pass cannot do without and `tolerance` how far two correct implementations may be apart.

Four kinds of pass:

  convolution     the message-passing convolution on a radius graph: `forward` (inference without
                  forces), `gradients` (forward and VJP: a training step on energies, or the forces
                  of a model) or `second` (forward, VJP and the VJP of the VJP: a training step on
                  forces), in both layouts and the three value types
  energy_forces   energy and forces of the two-layer model (molecular dynamics)
  tensor_product  the row-wise tensor product, forward and VJP
  radial_linear   the last layer of the radial network, forward and both gradients
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

import e3j_amd
from e3j_amd.harmonics import Harmonics
from e3j_amd.ops import prepare_graph
from e3j_amd.options import Layout, MixingMode
from e3j_amd.radial import radial_linear
from e3j_amd.workloads import EnergyModel, path_fan_in

CUTOFF = 5.0
DTYPES = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16}
#: node irreps, largest degree of the harmonics, output irreps: the tables the library is built for
TABLES = {
    "l1_l2_to_l2": ("0e+1o", 2, "0e+1o+2e"),
    "l2_l3_to_l2": ("0e+1o+2e", 3, "0e+1o+2e"),
    "l2_l3_to_l3": ("0e+1o+2e", 3, "0e+1o+2e+3o"),
    "l3_l3_to_l3": ("0e+1o+2e+3o", 3, "0e+1o+2e+3o"),
    "l0_l3_to_l3": ("0e", 3, "0e+1o+2e+3o"),
}
CHANNELS = {
    "l1_l2_to_l2": (32, 64, 128), "l2_l3_to_l2": (32, 64, 128), "l2_l3_to_l3": (64, 128),
    "l3_l3_to_l3": (32, 64, 128, 256), "l0_l3_to_l3": (64, 128, 256),
}


def _convolution(name, table, channels, atoms, passes, *, dtype="f32", layout="TRAILING_CHANNELS",
                 ordering="RECEIVER", graph="open", prepared=False, neighbours=30.0):
    """`graph`: "open" (a molecule or cluster), "periodic" (a box of liquid or solid) or "hubs" (a tenth
    of the nodes has six times the edges of the rest); `prepared`: the adjacency is kept over calls."""
    return dict(name=name, op="convolution", table=table, channels=channels, atoms=atoms, passes=passes,
                dtype=dtype, layout=layout, ordering=ordering, graph=graph, prepared=prepared,
                neighbours=neighbours)


def listed() -> list:
    return [
        # one small molecule, evaluated as it moves: the neighbour list is new in every call and the
        # pass is nothing but latency
        _convolution("molecule_forward", "l1_l2_to_l2", 32, 21, "forward"),
        # training step on a batch of small molecules (1 000 atoms, 32 channels): every batch has a graph
        # of its own, launches and host work count
        _convolution("batch_gradients", "l1_l2_to_l2", 32, 1000, "gradients"),
        # a layer of a mid-sized model on a box of 5 000 atoms (150k edges, 64 channels)
        _convolution("layer_gradients", "l2_l3_to_l2", 64, 5000, "gradients", graph="periodic"),
        # the large layer: 32 000 atoms, 0.96 M edges, 128 channels, degrees up to 3
        _convolution("large_gradients", "l3_l3_to_l3", 128, 32000, "gradients", graph="periodic"),
        # a graph that is not a radius graph: edges in any order, hub nodes, an odd number of nodes
        _convolution("hubs_gradients", "l2_l3_to_l2", 64, 4999, "gradients", ordering="NONE", graph="hubs"),
        # arrays kept channels-first, the layers of a model share the prepared graph
        _convolution("leading_gradients", "l3_l3_to_l3", 64, 10007, "gradients", layout="LEADING_CHANNELS",
                     graph="periodic", prepared=True),
        # half-precision training of the large layer
        _convolution("half_gradients", "l3_l3_to_l3", 128, 16000, "gradients", dtype="f16", graph="periodic",
                     prepared=True),
        # double precision, for reference data and stiff dynamics
        _convolution("double_gradients", "l3_l3_to_l3", 64, 8000, "gradients", dtype="f64", graph="periodic"),
        # training on forces: the loss is a function of the gradients of the layer
        _convolution("force_training", "l3_l3_to_l3", 128, 4000, "second", graph="periodic", prepared=True),
        # a step of molecular dynamics: energy and forces of two layers
        dict(name="energy_forces", op="energy_forces", atoms=6000, channels=64, hidden=32, l_max=3),
        # products of two feature arrays row by row (symmetric contractions of node features)
        dict(name="tensor_product", op="tensor_product", table="l3_l3_to_l3", rows=65537, channels=128,
             mode="MAP", dtype="f32", layout="TRAILING_CHANNELS"),
        # the last layer of a radial network of width 64 over 250k edges, 23 paths of 128 channels
        dict(name="radial_linear", op="radial_linear", edges=250007, hidden=64, width=2944),
    ]


def draw(rng) -> dict:
    """A case of the ranges that the listed ones stand for."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["convolution"] * 8 + ["energy_forces", "tensor_product", "radial_linear"])
    if kind == "energy_forces":
        # (the box has to hold two cutoffs)
        return dict(op=kind, atoms=spread(200, 8000), channels=rng.choice([64, 128]), hidden=rng.choice([16, 32, 64]),
                    l_max=rng.choice([2, 3]))
    if kind == "tensor_product":
        table, channels = rng.choice([("l2_l3_to_l3", 64), ("l2_l3_to_l3", 128), ("l3_l3_to_l3", 64),
                                      ("l3_l3_to_l3", 128)])
        dtype = rng.choice(["f32", "f32", "f64", "f16"])
        layout = rng.choice(["TRAILING_CHANNELS", "LEADING_CHANNELS"]) if dtype == "f32" else "TRAILING_CHANNELS"
        return dict(op=kind, table=table, rows=spread(500, 80_000), channels=channels,
                    mode=rng.choice(["MAP", "OUTER", "INNER"]), dtype=dtype, layout=layout)
    if kind == "radial_linear":
        hidden = rng.choice([8, 16, 32, 64, 128])
        return dict(op=kind, edges=spread(500, 40_000_000 // (hidden + 64)), hidden=hidden,
                    width=32 * rng.randint(8, 92))
    passes = rng.choice(["forward", "gradients", "gradients", "second"])
    table = rng.choice(sorted(TABLES))
    dtype = rng.choice(["f32", "f32", "f32", "f64", "f16"]) if passes != "second" else "f32"
    layout = "TRAILING_CHANNELS"
    if dtype == "f32" and passes != "second" and rng.random() < 0.25:
        layout = "LEADING_CHANNELS"
    channels = rng.choice([k for k in CHANNELS[table] if dtype == "f32" or k % 64 == 0])
    graph = rng.choice(["open", "periodic", "periodic", "hubs"])
    # at most the largest listed case's time: its 32 000 atoms at 128 channels, fewer for the slower passes
    most = {"f32": 32000, "f64": 8000, "f16": 24000}[dtype] * 128 // channels
    if passes == "second":
        most //= 8
    if layout == "LEADING_CHANNELS":
        most //= 2
    atoms = spread(12 if graph == "open" else 80, min(most, 40000))
    return _convolution(None, table, channels, atoms, passes, dtype=dtype, layout=layout,
                        ordering="NONE" if graph == "hubs" else rng.choice(["RECEIVER", "RECEIVER", "NONE"]),
                        graph=graph, prepared=rng.random() < 0.5,
                        neighbours=float(rng.choice([14, 22, 30]))) | {"name": ""}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Random:
    """Seeded values in GPU memory (every call draws from one generator, in program order)."""

    def __init__(self, seed: int):
        self.host = np.random.default_rng(seed)
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def uniform(self, *shape):
        return torch.rand(shape, dtype=torch.float64, device="cuda", generator=self.gen)

    def normal(self, *shape, dtype=torch.float32):
        return torch.randn(shape, dtype=dtype, device="cuda", generator=self.gen)

    def permutation(self, n: int):
        return torch.randperm(n, device="cuda", generator=self.gen)


def _box(atoms: int, neighbours: float) -> float:
    return (atoms / neighbours * 4.0 / 3.0 * math.pi * CUTOFF ** 3) ** (1.0 / 3.0)


def _edges(case) -> int:
    """Number of directed edges: what a cutoff of 5 gives on average."""
    n, mean = case["atoms"], case.get("neighbours", 30.0)
    if case.get("graph") == "hubs":
        return int(_hub_degrees(case).sum())
    box = _box(n, mean)
    if case.get("graph") == "open" or box <= 2.0 * CUTOFF:
        r = CUTOFF / box   # share of the pairs of random points of a cube that are closer than the cutoff
        share = 1.0 if r >= 1.0 else 4.0 / 3.0 * math.pi * r ** 3 - 1.5 * math.pi * r ** 4 + 1.6 * r ** 5 - r ** 6 / 6.0
        return max(2, int(n * (n - 1) * share) // 2 * 2)
    return int(n * mean) // 2 * 2


def _radius_graph(positions: torch.Tensor, box: float, periodic: bool, edges: int):
    """The `edges` shortest directed edges, i.e. a radius graph whose cutoff is set so that the number of
    edges does not depend on the seed; sorted by receiver, with the vectors sender - receiver."""
    n = positions.shape[0]
    periodic = periodic and box > 2.0 * CUTOFF
    reach = 1.25 * CUTOFF if n > 500 else math.inf   # candidates, of which the shortest are kept
    receivers, senders, lengths = [], [], []
    for first in range(0, n, 1024):
        delta = positions[None, :, :].float() - positions[first:first + 1024, None, :].float()
        if periodic:
            delta -= box * torch.round(delta / box)
        length = (delta * delta).sum(-1)
        rows = torch.arange(length.shape[0], device=length.device)
        near = length < reach ** 2
        near[rows, rows + first] = False
        r, s = near.nonzero(as_tuple=True)
        lengths.append(length[r, s])
        receivers.append(r + first)
        senders.append(s)
    receiver, sender = torch.cat(receivers), torch.cat(senders)
    keep = torch.sort(torch.cat(lengths), stable=True).indices[:edges].sort().values
    sender, receiver = sender[keep], receiver[keep]
    vec = positions[sender] - positions[receiver]
    shift = -box * torch.round(vec / box) if periodic else torch.zeros_like(vec)
    return sender.to(torch.int32), receiver.to(torch.int32), vec + shift, shift


def _hub_degrees(case) -> np.ndarray:
    """A tenth of the nodes receives six times the edges of the others; a quarter of spread around both."""
    n = case["atoms"]
    few = case["neighbours"] / 1.5
    degrees = few * np.linspace(0.75, 1.25, n)
    degrees[::10] *= 6
    return np.maximum(np.rint(degrees), 1).astype(np.int64)


def _hub_graph(case, rng: _Random):
    """Senders of the hubs come from two fifths of the nodes, of the other nodes from all of them."""
    n = case["atoms"]
    degree = torch.from_numpy(_hub_degrees(case)).cuda()[rng.permutation(n)]
    hub = degree > 2 * case["neighbours"]
    pool = rng.permutation(n)[: max(4, 2 * n // 5)]
    receiver = torch.repeat_interleave(torch.arange(n, device="cuda"), degree)
    pick = rng.uniform(receiver.shape[0])
    sender = torch.where(hub[receiver], pool[(pick * pool.shape[0]).long()], (pick * n).long())
    if case["ordering"] == "NONE":
        shuffle = rng.permutation(receiver.shape[0])
        sender, receiver = sender[shuffle], receiver[shuffle]
    return sender.to(torch.int32), receiver.to(torch.int32), rng.normal(receiver.shape[0], 3, dtype=torch.float64)


def _harmonics_irreps(l_max: int) -> str:
    return "+".join(f"{l}{'e' if l % 2 == 0 else 'o'}" for l in range(l_max + 1))


@functools.lru_cache(maxsize=None)
def _module(table: str, layout: str, ordering: str, neighbours: float):
    x_irreps, l_max, out_irreps = TABLES[table]
    return e3j_amd.Convolution((x_irreps, _harmonics_irreps(l_max)), out_irreps, graph_ordering=ordering,
                               layout=Layout.parse(layout), avg_num_neighbors=neighbours)


def _prepare_convolution(case, seed):
    rng = _Random(seed)
    module = _module(case["table"], case["layout"], case["ordering"], case["neighbours"])
    n, dtype, channels = case["atoms"], DTYPES[case["dtype"]], case["channels"]
    if case["graph"] == "hubs":
        sender, receiver, vec = _hub_graph(case, rng)
    else:
        box = _box(n, case["neighbours"])
        sender, receiver, vec, _ = _radius_graph(box * rng.uniform(n, 3), box, case["graph"] == "periodic",
                                                  _edges(case))
        if case["ordering"] == "NONE":
            shuffle = rng.permutation(sender.shape[0])
            sender, receiver, vec = sender[shuffle], receiver[shuffle], vec[shuffle]
    edges = sender.shape[0]
    num_x, num_z, num_s = module.source[0].dim, module.target.dim, module.params.num_scalars
    y = Harmonics(TABLES[case["table"]][1], normalization="component")(vec / vec.norm(dim=-1, keepdim=True)).to(dtype)
    leading = case["layout"] == "LEADING_CHANNELS"
    std = torch.from_numpy(1.0 / np.sqrt(path_fan_in(module))).to("cuda", dtype)

    def rows(count, dim, scale=None):
        shape = (count, channels, dim) if leading else (count, dim, channels)
        t = rng.normal(*shape, dtype=dtype)
        return t if scale is None else t.mul_(scale if leading else scale[:, None])

    state = dict(op=case["op"], passes=case["passes"], module=module, sender=sender, receiver=receiver,
                 x=rows(n, num_x), y=y, s=rows(edges, num_s, std), dm=rows(n, num_z),
                 graph=prepare_graph(sender, receiver, n, module.graph_ordering) if case["prepared"] else None)
    if case["passes"] == "second":   # cotangents of the gradients, as a loss on the forces sends them back
        state["cotangents"] = (rows(n, num_x), rng.normal(edges, y.shape[1], dtype=dtype), rows(edges, num_s, std))
    if case["passes"] != "forward":
        for t in ("x", "y", "s"):
            state[t].requires_grad_(True)
    if case["passes"] == "second":
        state["dm"].requires_grad_(True)
    return state


def _prepare_energy_forces(case, seed):
    rng = _Random(seed)
    irreps = _harmonics_irreps(case["l_max"])
    model = EnergyModel(channels=case["channels"], irreps=irreps, l_max=case["l_max"], hidden=case["hidden"],
                        cutoff=CUTOFF)
    n = case["atoms"]
    box = _box(n, 30.0)
    positions = box * rng.uniform(n, 3)
    sender, receiver, _, shift = _radius_graph(positions, box, True, _edges(case))
    return dict(op=case["op"], model=model, positions=positions.float(), shift=shift.float(), sender=sender,
                receiver=receiver, features=rng.normal(n, model.num_x, case["channels"]))


@functools.lru_cache(maxsize=None)
def _product(table: str, mode: str, layout: str):
    x_irreps, l_max, out_irreps = TABLES[table]
    return e3j_amd.TensorProduct((x_irreps, _harmonics_irreps(l_max)), out_irreps, mode=MixingMode[mode],
                                 layout=Layout.parse(layout))


def _prepare_tensor_product(case, seed):
    rng = _Random(seed)
    product = _product(case["table"], case["mode"], case["layout"])
    dtype, rows, channels = DTYPES[case["dtype"]], case["rows"], case["channels"]
    leading = case["layout"] == "LEADING_CHANNELS"

    def array(dim, k):
        shape = (rows, dim) if k == 0 else (rows, k, dim) if leading else (rows, dim, k)
        return rng.normal(*shape, dtype=dtype)

    num_x, num_y = (s.dim for s in product.source)
    # (OUTER: node features times one harmonics row per edge; INNER: channels summed)
    y = array(num_y, 0 if case["mode"] == "OUTER" else channels)
    dz = array(product.target.dim, 0 if case["mode"] == "INNER" else channels)
    return dict(op=case["op"], product=product, x=array(num_x, channels).requires_grad_(True),
                y=y.requires_grad_(True), dz=dz)


def _prepare_radial_linear(case, seed):
    rng = _Random(seed)
    h = torch.nn.functional.silu(rng.normal(case["edges"], case["hidden"]))
    w = rng.normal(case["hidden"], case["width"]) / math.sqrt(case["hidden"])
    return dict(op=case["op"], h=h.requires_grad_(True), w=w.requires_grad_(True),
                ds=rng.normal(case["edges"], case["width"]))


def prepare(case, seed):
    return {"convolution": _prepare_convolution, "energy_forces": _prepare_energy_forces,
            "tensor_product": _prepare_tensor_product, "radial_linear": _prepare_radial_linear}[case["op"]](case, seed)


# ---------------------------------------------------------------------------
# passes
# ---------------------------------------------------------------------------
def _run_convolution(state):
    x, y, s = state["x"], state["y"], state["s"]
    out = state["module"](x, y, s, state["sender"], state["receiver"], graph=state["graph"])
    if state["passes"] == "forward":
        return {"out": out}
    if state["passes"] == "gradients":
        dx, dy, ds = torch.autograd.grad(out, (x, y, s), state["dm"])
        return {"out": out.detach(), "dx": dx, "dy": dy, "ds": ds}
    dx, dy, ds = torch.autograd.grad(out, (x, y, s), state["dm"], create_graph=True)
    d2x, d2y, d2s, d2dm = torch.autograd.grad((dx, dy, ds), (x, y, s, state["dm"]), state["cotangents"])
    return {"out": out.detach(), "dx": dx.detach(), "dy": dy.detach(), "ds": ds.detach(),
            "d2x": d2x, "d2y": d2y, "d2s": d2s, "d2dm": d2dm}


def run(state):
    if state["op"] == "convolution":
        return _run_convolution(state)
    if state["op"] == "energy_forces":
        energy, forces = state["model"].energy_and_forces(state["positions"], state["features"], state["sender"],
                                                          state["receiver"], state["shift"])
        return {"energy": energy, "forces": forces}
    if state["op"] == "tensor_product":
        z = state["product"](state["x"], state["y"])
        dx, dy = torch.autograd.grad(z, (state["x"], state["y"]), state["dz"])
        return {"z": z.detach(), "dx": dx, "dy": dy}
    s = radial_linear(state["h"], state["w"])
    dh, dw = torch.autograd.grad(s, (state["h"], state["w"]), state["ds"])
    return {"s": s.detach(), "dh": dh, "dw": dw}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _work_convolution(case):
    module = _module(case["table"], case["layout"], case["ordering"], case["neighbours"])
    n, e, k = case["atoms"], _edges(case), case["channels"]
    size = DTYPES[case["dtype"]].itemsize
    nx, ny, nz, ns = (module.source[0].dim, module.source[1].dim, module.target.dim, module.params.num_scalars)
    x, y, s, z = n * nx * k, e * ny, e * ns * k, n * nz * k
    index = 4 * (2 * e)
    # a multiply-add per coefficient and channel for the messages, one for each of the gradients
    ops = 2.0 * e * k * len(module.coef.val)
    moved, passes = (x + y + s + z) * size + index, ops
    if case["passes"] in ("gradients", "second"):
        moved += (2 * (x + y + s) + z) * size + index
        passes += 3 * ops
    if case["passes"] == "second":
        # reads x, y, s, dm and three cotangents, writes four gradients; each gradient is two or three products
        moved += (3 * (x + y + s) + 2 * z) * size + index
        passes += 9 * ops
    return {"bytes": moved, "flops": passes}


def _work_energy_forces(case):
    n, k = case["atoms"], case["channels"]
    e = _edges(case)
    total, ops = 0.0, 0.0
    irreps = _harmonics_irreps(case["l_max"])
    module = e3j_amd.Convolution((irreps, irreps), irreps, graph_ordering="RECEIVER", avg_num_neighbors=30.0)
    nx, ny, nz, ns = (module.source[0].dim, module.source[1].dim, module.target.dim, module.params.num_scalars)
    for layer in range(2):
        # the hidden layer in, its cotangent out, node features and messages each way
        total += 4 * (2 * e * case["hidden"] + 2 * e * ny + 2 * n * nx * k + 2 * n * nz * k)
        # the radial weights, as they cross the convolution's boundary: written and read by the forward pass,
        # read again by the backward, whose gradient is written and read
        total += 4 * 5 * e * ns * k
        ops += 2.0 * e * k * (4 * len(module.coef.val) + 2 * case["hidden"] * ns)
        ops += 4.0 * n * nz * k * k
    return {"bytes": total + 4 * e * 10, "flops": ops}


def _work_tensor_product(case):
    product = _product(case["table"], case["mode"], case["layout"])
    k, r = case["channels"], case["rows"]
    x = r * product.source[0].dim * k
    y = r * product.source[1].dim * (1 if case["mode"] == "OUTER" else k)
    z = r * product.target.dim * (1 if case["mode"] == "INNER" else k)
    return {"bytes": DTYPES[case["dtype"]].itemsize * (3 * x + 3 * y + 2 * z),
            "flops": 6.0 * r * k * len(product.values)}


def _work_radial_linear(case):
    e, h, w = case["edges"], case["hidden"], case["width"]
    return {"bytes": 4.0 * (2 * e * w + 3 * e * h + 3 * h * w), "flops": 6.0 * e * h * w}


def work(case):
    return {"convolution": _work_convolution, "energy_forces": _work_energy_forces,
            "tensor_product": _work_tensor_product, "radial_linear": _work_radial_linear}[case["op"]](case)


def tolerance(case):
    """Relative error in the 2-norm: about four times what the passes show against the same pass in
    64 bits (float64: against its own sums in another order, in units of its last place)."""
    if case["op"] == "energy_forces":    # forces 7e-7; the energy is a sum over atoms that cancels in part
        return {"rel": 1e-5}
    if case["op"] == "radial_linear":    # 1.4e-6: the weight gradient sums over all edges
        return {"rel": 5e-6}
    # float32: 1.5e-7; float16: 9e-4 (node gradients are summed in half, in an order that changes from run to run)
    return {"rel": {"f32": 6e-7, "f64": 1.2e-15, "f16": 4e-3}[case["dtype"]]}
