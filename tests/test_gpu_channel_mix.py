"""`ChannelMix` in the matrix-core kernel: sums of split products against float64, tile and chunk edges, values whose
sizes differ from row to row, along the sums and against each other, and values that are no numbers."""

import numpy as np
import pytest
import torch

from e3j_amd import ChannelMix
from oracle import edge_oracle as E

pytestmark = pytest.mark.gpu


def _run(out, blocks, K, weights, dx=None):
    mixer = ChannelMix(blocks, K, weights)
    o = torch.as_tensor(out, device="cuda").float().requires_grad_(True)
    x = mixer(o)
    if dx is None:
        return x.detach().cpu().double().numpy()
    (g,) = torch.autograd.grad(x, o, torch.as_tensor(dx, device="cuda").float())
    return x.detach().cpu().double().numpy(), g.cpu().double().numpy()


def _problem(n, blocks, K, seed=0):
    rng = np.random.default_rng(seed)
    exact = lambda a: a.astype(np.float32).astype(np.float64)   # noqa: E731
    out = exact(rng.normal(size=(n, sum(m * d for m, d in blocks), K)))
    dx = exact(rng.normal(size=(n, sum(d for _, d in blocks), K)))
    return out, dx, [exact(rng.normal(size=(m, K, K))) for m, _ in blocks]


def _bound(got, want, sizes):
    """Six in 2^24 of a term (its six partial products are added in float32, what is left out is 2^-26 of it) and a
    rounding of 2^-24 per addition; `sizes`: the same sums of the terms' magnitudes, `terms` of them through at most 60 additions."""
    return np.abs(got - want) <= (6 + 60) * 2.0 ** -24 * sizes


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("n,blocks", [(1, [(1, 1)]), (31, [(2, 1), (1, 3)]), (33, [(1, 1), (3, 5)]), (127, [(1, 1)]),
                                      (129, [(4, 1), (7, 3)])])
@pytest.mark.parametrize("scales", ["one", "rows", "columns", "chunks", "opposed 8", "opposed 14", "opposed 20",
                                    "opposed 40"])
def test_against_float64(K, n, blocks, scales):
    out, dx, weights = _problem(n, blocks, K)
    if scales == "rows":         # nodes 2^60 apart, and a node of zeros
        out *= 2.0 ** (np.arange(n) % 7 * 10 - 30)[:, None, None]
        dx *= 2.0 ** (np.arange(n) % 5 * 10 - 20)[:, None, None]
        out[n // 2], dx[n // 2] = 0.0, 0.0
    elif scales == "columns":    # of the weights either way (the backward's columns are their rows)
        weights = [w * 2.0 ** (np.arange(K) % 5 * 9 - 18)[None, None, :] * 2.0 ** (np.arange(K) % 3 * 9)[None, :, None]
                   for w in weights]
    elif scales == "chunks":     # copies and halves of a row that differ by orders of magnitude
        weights = [w * 2.0 ** (np.arange(w.shape[0]) * 12)[:, None, None] for w in weights]
        out[..., K // 2:] *= 2.0 ** 20
        dx[..., K // 2:] *= 2.0 ** -20
    elif scales.startswith("opposed"):   # terms of a size, whose factors differ by orders of magnitude along both sums
        rng, bits = np.random.default_rng(n), int(scales.split()[1])
        plain, mixed = (2.0 ** rng.integers(-bits, bits + 1, K) for _ in range(2))
        out, dx = out * plain, dx * mixed
        weights = [w / plain[None, :, None] / mixed[None, None, :] for w in weights]
    x, g = _run(out, blocks, K, weights, dx)
    sizes = E.channel_mix(np.abs(out), blocks, [np.abs(w) for w in weights])
    assert _bound(x, E.channel_mix(out, blocks, weights), sizes).all()
    sizes = E.channel_mix_vjp(np.abs(dx), blocks, [np.abs(w) for w in weights])
    assert _bound(g, E.channel_mix_vjp(dx, blocks, weights), sizes).all()


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("blocks", [[(1, 1)], [(9, 1)], [(4, 1), (2, 3)]])
def test_errors_of_sums_of_one_size(K, blocks):
    """Normal values: a sum of k parts of random sign, rounded (or cut off) after each, is 2^-24 sqrt((k + 1) / 2) off, rms,
    beside the rounding of the parts; a part is a chunk of 64 channels."""
    out, dx, weights = _problem(500, blocks, K)
    x, g = _run(out, blocks, K, weights, dx)
    for got, want, parts in ((x, E.channel_mix(out, blocks, weights), max(m for m, _ in blocks) * K // 64),
                             (g, E.channel_mix_vjp(dx, blocks, weights), K // 64)):
        error = np.sqrt(((got - want) ** 2).mean() / (want ** 2).mean())
        assert error <= 2.0 ** -24 * np.sqrt((parts + 1) / 2 + 1), error


@pytest.mark.parametrize("K", [64, 128])
def test_weights_that_pick_one_channel(K):
    """One term a sum, beside channels of any size: the six partial products of that term, added in float32, and 2^-26
    of it left out."""
    blocks, n = [(1, 1), (1, 3)], 70
    out, dx, weights = _problem(n, blocks, K)
    out *= 2.0 ** np.random.default_rng(0).integers(-60, 61, K)
    dx *= 2.0 ** np.random.default_rng(1).integers(-60, 61, K)
    weights = [np.where(np.eye(K)[None] > 0, w, 0.0) for w in weights]
    x, g = _run(out, blocks, K, weights, dx)
    for got, want in ((x, E.channel_mix(out, blocks, weights)), (g, E.channel_mix_vjp(dx, blocks, weights))):
        assert (np.abs(got - want) <= 6.25 * 2.0 ** -24 * np.abs(want)).all()


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("small", ["row", "weights"])
def test_operands_whose_last_bits_leave_the_range_of_a_part(K, small):
    """Near 2^-120 the lowest of three bfloat16 parts would lie below the smallest bfloat16."""
    blocks, n = [(2, 1)], 40
    out, dx, weights = _problem(n, blocks, K)
    if small == "row":
        out[7, :, K // 2:] *= 2.0 ** -121
        out[7, :, :K // 2], dx[7] = 0.0, dx[7] * 2.0 ** -120
    else:
        weights = [w * 2.0 ** -120 for w in weights]
    out, dx, weights = (np.asarray(a, np.float32).astype(np.float64) for a in (out, dx, weights[0]))
    x, g = _run(out, blocks, K, [weights], dx)
    sizes = E.channel_mix(np.abs(out), blocks, [np.abs(weights)])
    assert _bound(x, E.channel_mix(out, blocks, [weights]), sizes).all()
    sizes = E.channel_mix_vjp(np.abs(dx), blocks, [np.abs(weights)])
    assert _bound(g, E.channel_mix_vjp(dx, blocks, [weights]), sizes).all()


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_that_are_no_numbers_stay_where_they_belong(K, bad):
    blocks, n = [(1, 1), (2, 3)], 70
    out, dx, weights = _problem(n, blocks, K)
    clean = _run(out, blocks, K, weights, dx)
    out[40, 1 + 3, 5], dx[41, 2, 7] = bad, bad    # copy 1, component 0 of the second degree; its component 1
    x, g = _run(out, blocks, K, weights, dx)
    assert np.isfinite(np.delete(x.reshape(n * 4, K), 40 * 4 + 1, 0)).all()
    want = bad * np.sign(weights[1][1, 5])
    assert np.array_equal(x[40, 1], want, equal_nan=True)
    for u in range(2):
        assert np.array_equal(g[41, 1 + 3 * u + 1], bad * np.sign(weights[1][u, :, 7]), equal_nan=True)
        g[41, 1 + 3 * u + 1] = clean[1][41, 1 + 3 * u + 1]
    assert np.isfinite(g).all()
    np.testing.assert_allclose(np.delete(x.reshape(n * 4, K), 161, 0), np.delete(clean[0].reshape(n * 4, K), 161, 0),
                               rtol=0, atol=128 * 2.0 ** -24 * 2 * K)   # (a tile beside it may take the other way)
    out, dx, weights = _problem(n, blocks, K)
    weights[1][0, 3, 9] = bad                     # a column of one degree
    x = _run(out, blocks, K, weights)
    assert np.array_equal(x[:, 1:, 9], bad * np.sign(out[:, 1:4, 3]), equal_nan=True)
    x[:, 1:, 9] = 0
    assert np.isfinite(x).all()


@pytest.mark.parametrize("K", [64, 128])
def test_the_ends_of_the_range(K):
    """Rows near the largest float with weights near the smallest: the sum fits, scaled operands do as well."""
    blocks, n = [(1, 1)], 5
    out, dx, weights = _problem(n, blocks, K)
    out, weights = out / np.abs(out).max() * 2.0 ** 127, [weights[0] / np.abs(weights[0]).max() * 2.0 ** -120]
    x = _run(out, blocks, K, weights)
    assert _bound(x, E.channel_mix(out, blocks, weights), E.channel_mix(np.abs(out), blocks, [np.abs(weights[0])])).all()


def test_nodes_too_far_apart_for_one_launch():
    """More than 2^25 values a node: a launch a node."""
    K, n, dim = 64, 2, (1 << 25) // 64 + 1
    w = np.random.default_rng(3).normal(size=(1, K, K)).astype(np.float32)
    mixer = ChannelMix([(1, dim)], K, [w])
    g = torch.Generator(device="cuda").manual_seed(0)
    out = torch.randn(n, dim, K, device="cuda", generator=g, requires_grad=True)
    x = mixer(out)
    dx = torch.randn(x.shape, device="cuda", generator=g)
    (grad,) = torch.autograd.grad(x, out, dx)
    weights = torch.as_tensor(w[0], device="cuda")
    # the bound of `_bound` with the largest sum of magnitudes there is, for the products of torch as well
    for got, a, b in ((x.detach(), out.detach(), weights), (grad, dx, weights.t().contiguous())):
        want = (a.view(-1, K) @ b).view_as(got)
        size = float(a.abs().max()) * float(b.abs().sum(0).max())
        assert float((got - want).abs().max()) <= 2 * 66 * 2.0 ** -24 * size
