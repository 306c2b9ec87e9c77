"""The native call of a module (`e3j_amd/native.py`) against the Python operators it stands in for: the same
library calls, hence the same bits where the kernels have a fixed order, and the same derivatives, routes and errors."""

import contextlib
import copy
import threading

import pytest
import torch

import e3j_amd
from e3j_amd import _lib, native, ops
from e3j_amd.options import config

pytestmark = pytest.mark.gpu

#: differences that the order of the dx atomics makes (dx and half-precision dy rows), relative to the largest value
ROUNDING = {torch.float32: 3e-6, torch.float64: 1e-14, torch.float16: 2e-2}


def _operands(n=300, channels=64, dtype=torch.float32, layout="TRAILING_CHANNELS", ordering="RECEIVER", degree=12, seed=0,
              hub=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = e3j_amd.Convolution(("0e+1o", "0e+1o+2e"), "0e+1o+2e", graph_ordering=ordering, layout=layout,
                            avg_num_neighbors=float(degree))
    receiver = torch.arange(n, device="cuda", dtype=torch.int32).repeat_interleave(degree)
    if hub:
        receiver = torch.cat([torch.zeros(hub, device="cuda", dtype=torch.int32), receiver])
    e = receiver.numel()
    sender = torch.randint(0, n, (e,), device="cuda", generator=g, dtype=torch.int32)
    if ordering == "NONE":
        shuffle = torch.randperm(e, device="cuda", generator=g)
        sender, receiver = sender[shuffle], receiver[shuffle]

    def rows(count, dim):
        shape = (count, dim, channels) if layout == "TRAILING_CHANNELS" else (count, channels, dim)
        return torch.randn(shape, device="cuda", generator=g).to(dtype)

    x, s, dm = rows(n, m.source[0].dim), rows(e, m.params.num_scalars), rows(n, m.target.dim)
    y = torch.randn(e, m.source[1].dim, device="cuda", generator=g).to(dtype)
    m(x, y, s, sender, receiver)   # (the first call of a kind of operand is the Python operators')
    return m, [t.requires_grad_(True) for t in (x, y, s)], sender, receiver, dm


def _grads(m, xs, sender, receiver, dm, graph=None, **kw):
    out = m(*xs, sender, receiver, graph=graph)
    return (out.detach(), *torch.autograd.grad(out, xs, dm, **kw))


def _python(monkeypatch):
    monkeypatch.setattr(native, "call", lambda *a: None)


def _same(got, want, dtype):
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert bool((a - b).abs().max() <= ROUNDING[dtype] * b.abs().max())


@pytest.mark.parametrize("dtype,layout,channels", [
    (torch.float32, "TRAILING_CHANNELS", 32), (torch.float32, "TRAILING_CHANNELS", 64), (torch.float32, "LEADING_CHANNELS", 64),
    (torch.float64, "TRAILING_CHANNELS", 64), (torch.float16, "TRAILING_CHANNELS", 128)])
@pytest.mark.parametrize("ordering", ["RECEIVER", "NONE"])
@pytest.mark.parametrize("prepared", [False, True])
@pytest.mark.parametrize("n,hub", [(2, 0), (100, 0), (300, 900)])
def test_matches_the_python_operators(monkeypatch, dtype, layout, channels, ordering, prepared, n, hub):
    m, xs, sender, receiver, dm = _operands(n, channels, dtype, layout, ordering, hub=hub)
    graph = e3j_amd.ops.prepare_graph(sender, receiver, n, ordering) if prepared else None
    with monkeypatch.context() as patch:   # (neither way through the Python operators)
        patch.setattr(ops, "_apply_fwd", None)
        if not prepared:                   # (a handle's schedule is built by its first backward, in Python)
            patch.setattr(ops, "_apply_bwd", None)
        got = _grads(m, xs, sender, receiver, dm, graph)
    with monkeypatch.context() as patch:
        if prepared:
            patch.setattr(ops, "_apply_bwd", None)
        again = _grads(m, xs, sender, receiver, dm, graph)
    with torch.no_grad():
        alone = m(*xs, sender, receiver, graph=graph)
    _python(monkeypatch)
    want = _grads(m, xs, sender, receiver, dm, graph)
    _same(got, want, dtype)
    _same(again, want, dtype)
    assert torch.equal(alone, want[0]) and not alone.requires_grad


def test_float64_over_tiles(monkeypatch):
    """(the rule of sizes is the operators': a call of its own and a handle lie on either side of it)"""
    g = torch.Generator(device="cuda").manual_seed(1)
    m = e3j_amd.Convolution(("0e+1o+2e+3o", "0e+1o+2e+3o"), "0e+1o+2e+3o", graph_ordering="RECEIVER")
    n, degree, channels = 1100, 10, 64
    assert ops._tiles_pay_f64(n * degree, 16, 23, channels, True) and not ops._tiles_pay_f64(n * degree, 16, 23, channels, False)
    receiver = torch.arange(n, device="cuda", dtype=torch.int32).repeat_interleave(degree)
    sender = torch.randint(0, n, receiver.shape, device="cuda", generator=g, dtype=torch.int32)
    rows = lambda *shape: torch.randn(shape, device="cuda", dtype=torch.float64, generator=g)   # noqa: E731
    xs = [t.requires_grad_(True) for t in (rows(n, 16, channels), rows(n * degree, 16), rows(n * degree, 23, channels))]
    dm = rows(n, 99, channels)
    graph = ops.prepare_graph(sender, receiver, n)
    m(*xs, sender, receiver)
    first, kept, own = (_grads(m, xs, sender, receiver, dm, h) for h in (graph, graph, None))
    _python(monkeypatch)
    want = _grads(m, xs, sender, receiver, dm)
    for got in (first, kept, own):
        _same(got, want, torch.float64)


@pytest.mark.parametrize("prepared", [False, True])
def test_derivatives_of_derivatives_and_kept_graphs(monkeypatch, prepared):
    m, xs, sender, receiver, dm = _operands(64, 64)
    dm.requires_grad_(True)
    graph = e3j_amd.ops.prepare_graph(sender, receiver, 64) if prepared else None

    def second():
        out = m(*xs, sender, receiver, graph=graph)
        first = torch.autograd.grad(out, xs, dm, create_graph=True)
        again = torch.autograd.grad(out, xs, dm, retain_graph=True)   # the node runs twice
        sum(g.square().sum() for g in first).backward()
        grads = [t.grad.clone() for t in (*xs, dm)]
        for t in (*xs, dm):
            t.grad = None
        return [out.detach(), *(g.detach() for g in first), *again, *grads]

    got = second()
    _python(monkeypatch)
    _same(got, second(), torch.float32)


def test_hooks_strides_and_alignment(monkeypatch):
    m, xs, sender, receiver, dm = _operands(50, 64)
    want = _grads(m, xs, sender, receiver, dm)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.detach().cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda().mT.contiguous().mT if t.dim() == 3 else t.cuda()):
        out = m(*xs, sender, receiver)
    assert len(packed) == 3
    _same((out.detach(), *torch.autograd.grad(out, xs, dm)), want, torch.float32)
    # a cotangent that is expanded, strided or off a 16-byte boundary, and one that stays undefined
    total = m(*xs, sender, receiver).sum()
    ones = _grads(m, xs, sender, receiver, torch.ones_like(dm))
    _same((want[0], *torch.autograd.grad(total, xs)), (want[0], *ones[1:]), torch.float32)
    off = torch.zeros(dm.numel() + 1, device="cuda")[1:].view_as(dm).copy_(dm)
    _same(_grads(m, xs, sender, receiver, off), want, torch.float32)
    # operands that need a copy
    x = xs[0].detach().mT.contiguous().mT
    s = torch.zeros(xs[2].numel() + 1, device="cuda")[1:].view(xs[2].shape).copy_(xs[2].detach())
    assert torch.equal(m(x, xs[1].detach(), xs[2].detach(), sender, receiver), want[0])
    # (off a 16-byte boundary other kernels run, which sum in another order)
    torch.testing.assert_close(m(xs[0].detach(), xs[1].detach(), s, sender, receiver), want[0], rtol=1e-5, atol=1e-5)
    assert torch.equal(m(xs[0], xs[1], xs[2], sender.long(), receiver.long()).detach(), want[0])
    strided = torch.stack([sender, receiver], 1)
    assert torch.equal(m(*xs, strided[:, 0], strided[:, 1]).detach(), want[0])


def test_transforms_modes_and_errors():
    m, xs, sender, receiver, dm = _operands(40, 64)
    want = _grads(m, xs, sender, receiver, dm)
    plain = [t.detach() for t in xs]
    out, vjp = torch.func.vjp(lambda *a: m(*a, sender, receiver), *plain)
    _same((out, *vjp(dm)), want, torch.float32)
    batched = torch.func.vmap(lambda x: m(x, *plain[1:], sender, receiver))(torch.stack([plain[0], 2 * plain[0]]))
    torch.testing.assert_close(batched[1], 2 * want[0], rtol=1e-5, atol=1e-5)
    with torch.autograd.forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        dual = torch.autograd.forward_ad.make_dual(plain[0], torch.ones_like(plain[0]))
        torch.autograd.forward_ad.unpack_dual(m(dual, *plain[1:], sender, receiver)).tangent.sum().item()
    with torch.inference_mode():
        assert torch.equal(m(*plain, sender, receiver), want[0])
    other = ops.prepare_graph(sender, receiver, 41)
    with pytest.raises(ValueError, match="41 nodes"):
        m(*xs, sender, receiver, graph=other)
    unsorted = e3j_amd.Convolution(("0e+1o", "0e+1o+2e"), "0e+1o+2e", graph_ordering="NONE", avg_num_neighbors=12.0)
    with pytest.raises(ValueError, match="ordering"):
        unsorted(*xs, sender, receiver, graph=ops.prepare_graph(sender, receiver, 40))
    with pytest.raises(RuntimeError, match="GPU memory"):
        m(*(t.detach().cpu() for t in xs), sender.cpu(), receiver.cpu())
    with pytest.raises(AttributeError):
        m(plain[0].tolist(), *plain[1:], sender, receiver)
    assert m(plain[0], plain[1][:0], plain[2][:0], sender[:0], receiver[:0]).abs().max() == 0
    twin = copy.deepcopy(m)
    assert torch.equal(twin(*plain, sender, receiver), want[0])


@pytest.mark.parametrize("setting", [dict(deterministic=True), dict(tile_rows=0), dict(tile_rows=3), dict(row_cap=0),
                                     dict(row_cap=5), dict(fixed_order_rows=False), dict(locality_rounds=0),
                                     dict(locality_rounds=1), dict(pair_rows=True), dict(graph_cache=True)])
def test_settings(monkeypatch, setting):
    m, xs, sender, receiver, dm = _operands(500, 64, hub=700)
    with config.use(**setting):
        m(*xs, sender, receiver)
        got = _grads(m, xs, sender, receiver, dm)
        _python(monkeypatch)
        want = _grads(m, xs, sender, receiver, dm)
    ops.clear_graph_cache()
    if setting == dict(fixed_order_rows=False):   # (pieces added with atomics)
        torch.testing.assert_close(got[0], want[0], rtol=1e-5, atol=1e-5)
        got = (want[0], *got[1:])
    _same(got, want, torch.float32)


class _Calls:
    """The library with the names of the entries that the Python operators call on record."""

    def __init__(self, lib):
        self._lib, self.names = lib, []

    def __getattr__(self, name):
        if "convolution_bwd" in name:
            self.names.append(name)
        return getattr(self._lib, name)


@pytest.mark.parametrize("prepared", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_settings_of_the_backward(monkeypatch, dtype, prepared):
    """The backward follows the settings it runs under, not those of its forward call."""
    m, xs, sender, receiver, dm = _operands(300, 64, dtype)
    graph = ops.prepare_graph(sender, receiver, 300) if prepared else None
    want = _grads(m, xs, sender, receiver, dm, graph)
    native.load()
    lib = _Calls(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: lib)
    routes = {}
    for name, setting in (("deterministic", dict(deterministic=True)), ("tiles", dict(tile_rows=0)), ("same", None)):
        runs = []
        for _ in range(3):
            out = m(*xs, sender, receiver, graph=graph)
            with config.use(**setting) if setting else contextlib.nullcontext():
                runs.append((out.detach(), *torch.autograd.grad(out, xs, dm)))
            _same(runs[-1], want, dtype)
        if name == "deterministic":
            assert all(torch.equal(a, b) for r in runs[1:] for a, b in zip(r, runs[0]))
        routes[name] = list(lib.names)
        lib.names.clear()
    assert len(routes["deterministic"]) == len(routes["tiles"]) == 3 and not routes["same"]
    assert not any("tiled" in r for r in routes["deterministic"] + routes["tiles"])
    # the other way about: a forward pass of its own settings, the backward under the usual ones
    with config.use(tile_rows=0):
        m(*xs, sender, receiver, graph=graph)
        out = m(*xs, sender, receiver, graph=graph)
    _same((out.detach(), *torch.autograd.grad(out, xs, dm)), want, dtype)
    assert len(lib.names) == 1


def test_endpoints_beside_a_handle_are_refused_as_often_as_asked():
    m, xs, sender, receiver, _ = _operands(40, 64)
    graph = ops.prepare_graph(sender, receiver, 40)
    for _ in range(3):
        m(*xs, sender, receiver, graph=graph)
        for snd, rcv in ((sender.cpu(), receiver), (sender, receiver.cpu())):
            with pytest.raises(RuntimeError, match="GPU memory"):
                m(*xs, snd, rcv, graph=graph)
        with pytest.raises(TypeError, match="sender"):
            m(*xs, None, receiver, graph=graph)


def test_streams_and_threads():
    m, xs, sender, receiver, dm = _operands(400, 64)
    want = _grads(m, xs, sender, receiver, dm)
    graph = ops.prepare_graph(sender, receiver, 400)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for handle in (graph, None, graph):
            out = m(*xs, sender, receiver, graph=handle)
            grads = torch.autograd.grad(out, xs, dm)
            side.synchronize()
            _same((out.detach(), *grads), want, torch.float32)
        out = m(*xs, sender, receiver)
    torch.cuda.current_stream().wait_stream(side)
    _same((out.detach(), *torch.autograd.grad(out, xs, dm)), want, torch.float32)   # from another stream than the forward's
    torch.cuda.synchronize()
    failures = []

    def work(seed):
        try:
            mine = _operands(200 + seed, 64, seed=seed)
            with torch.cuda.stream(torch.cuda.Stream()):
                torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
                first = _grads(*mine)
                for _ in range(20):
                    again = _grads(*mine)
                torch.cuda.current_stream().synchronize()
                _same(again, first, torch.float32)
        except BaseException as e:   # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]


def test_forward_recorded_into_a_graph():
    m, xs, sender, receiver, _ = _operands(400, 64, ordering="RECEIVER", hub=300)
    x, y, s = (t.detach().clone() for t in xs)
    eager = m(x, y, s, sender, receiver)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m(x, y, s, sender, receiver)
    for scale in (1.0, 2.0, -0.5):
        x.copy_(xs[0].detach() * scale)
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(out, eager * scale, rtol=1e-6, atol=1e-6)
        torch.testing.assert_close(m(x, y, s, sender, receiver), out, rtol=0, atol=0)
