"""Leaf sets of more than 1,024 entries, which are kept as the low halves of their ids:
their numbers around the limits, ids in few buckets or in all, lists short enough to be
scanned or so long that the set's elements are searched in them, and graphs whose ids
have 16 bits below their bucket's or more."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SQUARE = np.array([(0, 1), (1, 2), (2, 3), (3, 0)], np.uint32)


def squares(n, fn, others, span, labels, seed):
    """Hub 0 with fn neighbours (the leaf set), hubs 1.. with `others` neighbours, all of
    them among `span` ids from the end of the graph, the even ones (of a label of their
    own, with two labels); hub 1's list holds the first and the last of hub 0's."""
    rng = np.random.default_rng(seed)
    ids = n - 1 - np.arange(0, 2 * span, 2)
    pa = np.sort(rng.choice(ids, fn, replace=False))
    lists = [pa] + [np.union1d(rng.choice(ids, k, replace=False), pa[[0, -1]]) for k in others]
    u = np.concatenate([np.full(len(p), h) for h, p in enumerate(lists)]).astype(np.uint32)
    v = np.concatenate(lists).astype(np.uint32)
    lab = np.zeros(n, np.uint32)
    lab[ids] = labels - 1
    query = (4, np.array([0, labels - 1] * 2, np.uint32), SQUARE[:, 0].copy(), SQUARE[:, 1].copy())
    src = np.array([0, 0, 1, 2], np.uint32)
    dst = np.array([pa[0], pa[-1], lists[1][len(lists[1]) // 2], lists[2][0]], np.uint32)
    return (n, lab, u, v), [query], (np.ones(4, np.uint8), src, dst, np.zeros(4, np.uint32))


def counts(graph, queries, batch, **kw):
    eng = E.Engine(graph, queries, relabel=False, **kw)
    try:
        pos, neg = eng.process_batch(*batch)
        return pos.tolist() + neg.tolist()
    finally:
        eng.close()


@pytest.mark.parametrize("fn", [1024, 1025, 1088, 1500, 2047, 2048])
@pytest.mark.parametrize("n,span", [(5000, 2100), (100000, 2100), (100000, 49000), (1 << 20, 500000)])
@pytest.mark.parametrize("labels", [1, 2])
def test_squares_over_long_leaf_sets(fn, n, span, labels):
    others = (min(1200, span), min(40000, span), min(2100, span))
    graph, queries, batch = squares(n, fn, others, span, labels, [fn, n, span, labels])
    want = O.run_stream(O.Graph(*graph), [O.Query(*queries[0])], [batch], relabel=False)[0]
    for kw in ({}, {"leaf_segments": False}, {"leaf_budget": 64}, {"leaf_budget": 0xFFFFFFFF}):
        assert counts(graph, queries, batch, **kw) == want["pos"] + want["neg"], kw


@pytest.mark.parametrize("n", [1 << 25, (1 << 25) + 1])
def test_ids_that_fill_a_half_and_that_pass_it(n):
    """The set in halves (or, past 2^25 vertices, not kept) counts what one descent per
    candidate counts, which uses no leaf set."""
    graph, queries, batch = squares(n, 1500, (1200, 40000, 2100), 16000000, 2, n)
    want = counts(graph, queries, batch, leaf_sets=False)
    assert any(want) and counts(graph, queries, batch) == want
