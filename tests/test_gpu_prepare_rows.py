"""Adjacency and tile schedule of a graph in few launches (`e3j_amd_prepare_rows`, the one-workgroup row
order and schedule) against numpy, at the sizes where a route ends: 256 rows (no order), 16 384 edges
(rows by one workgroup), 1 024 / 2 048 / 4 096 / 8 192 rows (order by one workgroup), 4 096 tiles."""

import numpy as np
import pytest
import torch

from e3j_amd.graph import TileSchedule, locality_order, prepare_rows

pytestmark = pytest.mark.gpu
DUMMY = 2 ** 31 - 1


def _rows(key, n):
    return np.concatenate([[0], np.cumsum(np.bincount(key[key != DUMMY], minlength=n))])


def _order(other, ptr, n):
    """Two sweeps of minimum labels over the first 128 positions of a row, rows sorted by (second, first)
    label, rows of more than twice the mean degree dealt to the fronts of eighths of the list."""
    labels = np.arange(n)
    levels = []
    for _ in range(2):
        new = labels.copy()
        for r in range(n):
            near = other[ptr[r]:min(ptr[r + 1], ptr[r] + 128)]
            near = near[near < n]
            if near.size:
                new[r] = min(new[r], labels[near].min())
        labels = new
        levels.append(new)
    rows = np.lexsort((np.arange(n), levels[0], levels[1]))
    long = (np.diff(ptr) * n > 2 * ptr[-1])[rows]
    longs, shorts, out = rows[long], rows[~long], []
    for p in range(8):
        out += [longs[p * len(longs) // 8:(p + 1) * len(longs) // 8],
                shorts[p * len(shorts) // 8:(p + 1) * len(shorts) // 8]]
    return np.concatenate(out)


def _graph(n, e, kind, seed):
    rng = np.random.default_rng(seed)
    key = np.sort(rng.integers(0, n, e))
    if kind == "hub":                       # one row of a third of the edges, most rows empty
        key = np.sort(np.where(rng.random(e) < 1 / 3, n // 2, rng.integers(0, max(1, n // 3), e)))
    other = rng.integers(0, n, e)
    other[rng.random(e) < 0.05] = DUMMY
    key[e - e // 10:] = DUMMY               # padding edges lie at the end
    return key.astype(np.int64), other.astype(np.int64)


@pytest.mark.parametrize("n,e,kind,form", [
    (1, 1, "even", "sorted"), (7, 3, "even", "sorted"), (256, 4000, "hub", "sorted"), (257, 4001, "even", "sorted"),
    (1000, 16384, "even", "sorted"), (1024, 16385, "hub", "sorted"), (1025, 20000, "even", "global"),
    (4096, 5000, "hub", "global"), (4097, 40000, "even", "mixed"), (300, 9000, "hub", "mixed"),
    (8192, 50000, "even", "sorted"), (8193, 50000, "hub", "sorted"), (1, 70, "even", "any"), (300, 5000, "hub", "any"),
    (5000, 60000, "even", "any"),
])
def test_against_numpy(n, e, kind, form):
    key, other = _graph(n, e, kind, n + e)
    rng = np.random.default_rng(e)
    given_key, given_other = key.copy(), other.copy()
    if form == "any":
        shuffle = rng.permutation(e)
        key, other = key[shuffle], other[shuffle]
        given_key, given_other = key.copy(), other.copy()
    if form == "mixed":                     # keys out of order although the call says sorted
        key = given_key = rng.permutation(key)
    if form == "global":                    # ids of another shard, reduced modulo the number of rows
        given_key = np.where(key == DUMMY, key, key - 3 * n)
        given_other = np.where(other == DUMMY, other, other + 2 * n)
    dev = lambda a: torch.from_numpy(a.astype(np.int32)).cuda()  # noqa: E731
    rounds = 2 if n > 256 else 0
    ptr, oth, perm, order, seg = prepare_rows(dev(given_key), dev(given_other), n, form != "any", rounds, (64, 64))
    want_ptr = _rows(key, n)
    np.testing.assert_array_equal(ptr.cpu().numpy(), want_ptr)
    if form == "any":
        want_perm = np.argsort(key, kind="stable")
        np.testing.assert_array_equal(perm.cpu().numpy(), want_perm)
        other = other[want_perm]
    else:
        assert perm is None
    np.testing.assert_array_equal(oth.cpu().numpy(), other)
    if rounds:
        np.testing.assert_array_equal(order.cpu().numpy(), _order(other, want_ptr, n))
    else:
        assert order is None
    listed = seg.buffer.cpu().numpy()
    got = listed[4:4 + 3 * listed[0]].reshape(-1, 3)
    want = [(r, b, min(b + 64, want_ptr[r + 1])) for r in range(n) if want_ptr[r + 1] - want_ptr[r] > 64
            for b in range(want_ptr[r] + 64, want_ptr[r + 1], 64)]
    assert sorted(map(tuple, got.tolist())) == want
    starts = got[np.flatnonzero(np.diff(got[:, 0], prepend=-1))][:, 0]
    assert len(set(starts.tolist())) == len(starts)      # the pieces of a row are adjacent


@pytest.mark.parametrize("n,e", [(16000, 16384), (9000, 16384), (40, 16384), (20000, 1000)])
def test_out_of_order_keys_of_one_workgroup(n, e):
    """Keys out of order in the route of one workgroup: its first pass writes row pointers that the count
    replaces, from other waves.  The first pass's stores are ordered before that (the kernel's fence), or one of
    them would overwrite a count."""
    rng = np.random.default_rng(n)
    dev = lambda a: torch.from_numpy(a.astype(np.int32)).cuda()  # noqa: E731
    for _ in range(20):
        key = rng.integers(0, n, e)
        key[rng.random(e) < 0.1] = DUMMY
        other = rng.integers(0, n, e)
        ptr, oth, _, _, _ = prepare_rows(dev(key), dev(other), n, True, 0)
        np.testing.assert_array_equal(ptr.cpu().numpy(), _rows(key, n))
        np.testing.assert_array_equal(oth.cpu().numpy(), other)


@pytest.mark.parametrize("n,tile_rows", [(1, 2), (4096, 1), (4097, 1), (8193, 2), (700, 8), (300, 65)])
def test_schedule_work_and_lists(n, tile_rows):
    e, max_work = 6 * n + 600, 64
    key, other = _graph(n, e, "hub" if n > 1 else "even", n)
    dev = lambda a: torch.from_numpy(a.astype(np.int32)).cuda()  # noqa: E731
    ptr, oth, _, _, _ = prepare_rows(dev(key), dev(other), n, True, 0)
    sch = TileSchedule(oth, ptr, None, None, n, tile_rows, max_work)
    ptr = ptr.cpu().numpy().astype(np.int64)
    tiles = -(-n // tile_rows)
    bounds = ptr[np.minimum(np.arange(tiles + 1) * tile_rows, n)]
    want = []
    for t in range(tiles):
        begin, end = bounds[t], bounds[t + 1]
        want += [(t, b, min(b + max_work, end)) for b in range(begin, end, max_work)] or [(t, begin, begin)]
    work = sch.work.cpu().numpy()
    assert work[0, 3] == len(want)
    np.testing.assert_array_equal(work[:len(want), :3], want)
    snd, edge, local = (v.cpu().numpy() for v in (sch.sender, sch.edge, sch.local))
    for t in range(tiles):
        pos = np.arange(bounds[t], bounds[t + 1])
        if not 0 < pos.size <= 512:
            continue
        s = np.where(other[pos] < n, other[pos], n)
        by = np.lexsort((pos, s))
        np.testing.assert_array_equal(snd[pos], np.where(s[by] == n, -1, s[by]))
        np.testing.assert_array_equal(edge[pos], pos[by])
        row = np.searchsorted(ptr, pos[by], side="right") - 1
        np.testing.assert_array_equal(local[pos], row - t * tile_rows)


@pytest.mark.parametrize("n,e,kind", [
    (1, 5, "even"), (300, 1024, "hub"), (300, 1025, "hub"), (2, 4095, "hub"), (3, 4096, "even"), (255, 4097, "even"), (256, 8192, "hub"), (8191, 12289, "hub"),
    (65535, 70001, "even"), (65536, 70001, "even"), (4999, 262144, "hub"), (4999, 262145, "even"), (40000, 262143, "even"),
])
def test_edge_sort_against_numpy(n, e, kind):
    """Unsorted edges at the sizes where the sort changes: 1 024 edges, digits of the keys, chunks of 4 096 edges, 64 of
    them, 2^16 nodes; ids of another shard and keys that are sorted already among them."""
    key, other = _graph(n, e, kind, n + e)
    shuffle = np.random.default_rng(e).permutation(e)
    dev = lambda a: torch.from_numpy(a.astype(np.int32)).cuda()  # noqa: E731
    for k, o in ((key[shuffle], other[shuffle]), (key, other)):
        shifted = np.where(k == DUMMY, k, k - 2 * n)
        ptr, oth, perm, order, _ = prepare_rows(dev(shifted), dev(o), n, False, 0, None)
        want = np.argsort(k, kind="stable")
        np.testing.assert_array_equal(perm.cpu().numpy(), want)
        np.testing.assert_array_equal(ptr.cpu().numpy(), _rows(k, n))
        np.testing.assert_array_equal(oth.cpu().numpy(), o[want])
        assert order is None


@pytest.mark.parametrize("kind", ["even", "hub"])
@pytest.mark.parametrize("n", [16384, 16385])
def test_row_order_either_side_of_four_lanes_a_row(n, kind):
    key, other = _graph(n, 5 * n, kind, n)
    dev = lambda a: torch.from_numpy(a.astype(np.int32)).cuda()  # noqa: E731
    ptr = _rows(key, n)
    order = locality_order(dev(other), dev(ptr), n, 2)
    np.testing.assert_array_equal(order.cpu().numpy(), _order(other, ptr, n))


def test_row_order_of_more_rows_than_a_sweep_has_threads():
    """2^27 rows and a few: sixteen lanes a row would be more than 2^31, and threads take several rows."""
    n = (1 << 27) + 9
    other = torch.arange(n, dtype=torch.int32, device="cuda")
    row_ptr = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    # (each row has itself for a neighbour, except three that belong to clusters at the front, one of them two hops away)
    far = [n - 1, 1 << 27, (1 << 26) + 3]
    other[far[0]], other[far[1]], other[far[2]] = 5, 100, n - 1
    order = locality_order(other, row_ptr, n, 2)
    del other, row_ptr
    front = [*range(6), far[0], far[2], *range(6, 101), far[1]]   # (labels 5, 5 and 100 after two sweeps)
    assert order[:len(front)].tolist() == front
    rest = order[len(front):]
    want = torch.arange(101, n, dtype=torch.int32, device="cuda")
    keep = torch.ones(n - 101, dtype=torch.bool, device="cuda")
    keep[torch.tensor([f - 101 for f in far], device="cuda")] = False
    assert torch.equal(rest, want[keep])
