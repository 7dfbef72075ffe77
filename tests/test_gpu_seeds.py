"""Seeding: the search for a record's edge at list lengths where it takes one step
more, few and many plans per record (more than a wave's queue of seeds holds), and
both shares of records per wave, against the oracle's counts."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

EDGES = {"edge": [(0, 1)], "path3": [(0, 1), (1, 2)], "triangle": [(0, 1), (1, 2), (0, 2)]}


def query(shape):
    e = np.array(EDGES[shape], np.uint32)
    return int(e.max()) + 1, np.zeros(int(e.max()) + 1, np.uint32), e[:, 0].copy(), e[:, 1].copy()


def check(graph, queries, batches):
    want = O.run_stream(O.Graph(*graph), [O.Query(*q) for q in queries], batches)
    eng = E.Engine(graph, queries)
    try:
        for i, b in enumerate(batches):
            pos, neg = eng.process_batch(*b)
            assert pos.tolist() == want[i]["pos"] and neg.tolist() == want[i]["neg"], i
    finally:
        eng.close()


@pytest.mark.parametrize("deg", [1, 15, 16, 17, 18, 272, 273, 288, 289, 290, 4914, 5000])
def test_edges_of_a_hub_are_found(deg):
    """Records on the first, last and middle entries of a list of `deg`, present or not."""
    n = 2 * deg + 3
    nbrs = np.arange(2, 2 * deg + 1, 2, dtype=np.uint32)  # the hub is 0, the odd vertices are not its neighbours
    graph = (n, np.zeros(n, np.uint32), np.zeros(deg, np.uint32), nbrs)
    at = np.unique(np.concatenate([nbrs[:20], nbrs[-20:], nbrs[:: max(1, deg // 37)], nbrs[:18] - 1]))
    zero = np.zeros(len(at), np.uint32)
    lab = np.zeros((len(at), 2), np.uint32)
    swap = np.arange(len(at)) % 2 == 0
    src, dst = np.where(swap, at, zero).astype(np.uint32), np.where(swap, zero, at).astype(np.uint32)
    batches = [(np.zeros(len(at), np.uint8), src, dst, lab[:, 0]), (np.ones(len(at), np.uint8), dst, src, lab[:, 0]),
               (np.zeros(len(at), np.uint8), dst, src, lab[:, 0])]
    check(graph, [query("edge"), query("path3")], batches)


@pytest.mark.parametrize("queries", [1, 3, 64])
@pytest.mark.parametrize("records", [1, 16, 17, 65, 300, 8192, 8193])
def test_many_plans_per_record(queries, records):
    """With 64 queries of one label a record has up to 320 plans."""
    n = 3 * records + 40
    rng = np.random.default_rng([queries, records])
    u, v = rng.integers(0, n, 2 * n).astype(np.uint32), rng.integers(0, n, 2 * n).astype(np.uint32)
    keep = u != v
    qs = [query(("triangle", "path3", "edge")[i % 3]) for i in range(queries)]
    add = rng.integers(0, 2, records).astype(np.uint8)
    src, dst = rng.integers(0, n + 2, records).astype(np.uint32), rng.integers(0, n, records).astype(np.uint32)
    src[src >= n] = dst[src >= n]  # some self-loops
    check((n, np.zeros(n, np.uint32), u[keep], v[keep]), qs, [(add, src, dst, np.zeros(records, np.uint32))])
