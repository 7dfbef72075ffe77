"""Refined candidates where a wave's work changes shape: 4,096 vertices to a wave,
64 candidates to a round, 64 entries to a list, 4,096 to a chunk."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = {"path3": [(0, 1), (1, 2)], "house": [(0, 1), (1, 2), (2, 3), (3, 0), (0, 4), (1, 4)],
          "combine_keep": [(0, 1), (4, 2), (3, 4), (3, 1), (1, 2), (0, 5), (0, 3)],
          "combine_late": [(1, 2), (0, 5), (0, 1), (1, 3), (2, 4), (0, 6), (5, 6)]}


@pytest.mark.parametrize("n,hub", [(n, hub) for n in (5, 63, 65, 4095, 4097, 8193)
                                   for hub in (0, 63, 64, 65, 4097, 8192) if hub < n])
@pytest.mark.parametrize("labels", [1, 2, 5])
def test_refined_candidates(n, hub, labels):
    rng = np.random.default_rng([n, labels, hub])
    m = 3 * n if labels > 1 else n
    u, v = rng.integers(0, n, m), rng.integers(0, n, m)
    u, v = np.concatenate([u, np.full(hub, 1)]), np.concatenate([v, rng.permutation(n)[:hub]])
    keep = u != v
    u, v = u[keep].astype(np.uint32), v[keep].astype(np.uint32)
    lab = rng.integers(0, labels, n).astype(np.uint32)
    queries = []
    for shape in SHAPES.values():
        e = np.array(shape, np.uint32)
        k = int(e.max()) + 1
        queries.append((k, rng.integers(0, labels, k).astype(np.uint32), e[:, 0].copy(), e[:, 1].copy()))
    g = O.Graph(n, lab, u, v)
    eng = E.Engine((n, lab, u, v), queries, cluster_filter=True)
    try:
        for qi, q in enumerate(queries):
            want = g.cluster_candidates(O.Query(*q))
            for x in range(q[0]):
                assert np.array_equal(eng.refined_candidates(qi, x), want[x].astype(bool)), (qi, x)
    finally:
        eng.close()
