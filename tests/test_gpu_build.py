"""The adjacency an engine makes of its edge list: order, duplicates, self-loops
and both directions at the sizes where its sort changes shape."""
import numpy as np
import pytest

from dsm_amd import engine as E

pytestmark = pytest.mark.gpu

EDGE = (2, np.zeros(2, np.uint32), np.zeros(1, np.uint32), np.ones(1, np.uint32))


def adjacency(n, u, v):
    keys = np.unique(np.concatenate([u.astype(np.uint64) << np.uint64(32) | v, v.astype(np.uint64) << np.uint64(32) | u]))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount((keys >> np.uint64(32)).astype(np.int64), minlength=n), out=off[1:])
    return off, (keys & np.uint64(0xFFFFFFFF)).astype(np.uint32)


def check(n, u, v):
    eng = E.Engine((n, np.zeros(n, np.uint32), u, v), [EDGE])
    try:
        off, nb, _ = eng.graph()
    finally:
        eng.close()
    want_off, want_nb = adjacency(n, u, v)
    assert np.array_equal(off, want_off) and np.array_equal(nb, want_nb)


# tiles of 2,048 edges, 16,384 edges to the second tile of the counts' scan
@pytest.mark.parametrize("m", [0, 1, 31, 2047, 2048, 2049, 16383, 16385, 70001])
@pytest.mark.parametrize("n", [1, 2, 256, 257, 65537])
def test_adjacency_of_random_edges(n, m):
    rng = np.random.default_rng([n, m])
    check(n, rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32))


@pytest.mark.parametrize("shape", ["star", "one_edge_many_times", "path_backwards"])
def test_adjacency_of_uneven_edges(shape):
    n = 70000
    a = np.arange(1, n, dtype=np.uint32)
    u, v = {"star": (np.full(n - 1, 5, np.uint32), a), "one_edge_many_times": (np.full(n, 9, np.uint32), np.full(n, 69999, np.uint32)),
            "path_backwards": (a[::-1].copy(), a[::-1] - 1)}[shape]
    check(n, u, v.astype(np.uint32))


def test_adjacency_past_one_round_of_the_scans_top():
    """More than 1,024 tiles in the scans of the counts and of the slots."""
    n, m = 2200000, 17000000
    rng = np.random.default_rng(7)
    check(n, rng.integers(0, n, m, dtype=np.uint32), rng.integers(0, n, m, dtype=np.uint32))


@pytest.mark.parametrize("at", [0, 1, 2047, 5000, 6999])
def test_first_edge_out_of_range_is_named(at):
    n, m = 300, 7000
    rng = np.random.default_rng(at)
    u, v = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    (u if at % 2 else v)[at] = n
    v[m - 1] = 0xFFFFFFFF
    with pytest.raises(E.DsmError, match="edge %d: endpoint out of range" % at):
        E.Engine((n, np.zeros(n, np.uint32), u, v), [EDGE])
