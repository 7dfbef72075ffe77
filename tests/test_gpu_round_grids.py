"""The grid of a DFS round: what the caller or the autotuner set, and what earlier rounds
of little work leave to heavy ones."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _mixed_graph():
    """6,000 vertices of 1,000 neighbours each beside 6,000 of two: (graph, queries,
    heavy batch, light batch), 400 inserts of edges that are there each."""
    n, rng = 6000, np.random.default_rng(4)
    i = np.arange(n)
    u = np.concatenate([np.repeat(i, 500), n + i])
    v = np.concatenate([(np.repeat(i, 500) + np.tile(rng.choice(np.arange(1, n // 2), 500, replace=False), n)) % n,
                        n + (i + 1) % n])
    graph = (2 * n, np.zeros(2 * n, np.uint32), u.astype(np.uint32), v.astype(np.uint32))
    sq = np.array([(0, 1), (1, 2), (2, 3), (3, 0)], np.uint32)
    pick = rng.choice(500 * n, 400, replace=False)
    heavy, light = ((np.ones(400, np.uint8), graph[2][p], graph[3][p], np.zeros(400, np.uint32))
                    for p in (pick, 500 * n + rng.choice(n, 400, replace=False)))
    return graph, [(4, np.zeros(4, np.uint32), sq[:, 0].copy(), sq[:, 1].copy())], heavy, light


def _waves(eng, batch):
    eng.process_batch(*batch)
    s = eng.stats()
    return s["dfs_waves"] // s["dfs_launches"]


def test_a_given_or_tuned_grid_is_kept():
    """Rounds of little work start as many blocks as the caller set, or dsm_autotune found."""
    graph, queries, _, light = _mixed_graph()
    eng = E.Engine(graph, queries, relabel=False, blocks_per_cu=3)
    try:
        waves = [_waves(eng, light) for _ in range(4)]
        assert len(set(waves)) == 1 and waves[0] % 12 == 0
        cus = waves[0] // 12
    finally:
        eng.close()
    eng = E.Engine(graph, queries, relabel=False)
    try:
        rep = eng.autotune(*light)
        want = rep["blocks_per_cu"] * rep["waves_per_block"] * cus
        assert [_waves(eng, light) for _ in range(4)] == [want] * 4
    finally:
        eng.close()


def test_light_rounds_leave_heavy_ones_their_grid():
    """Rounds of heavy records among light ones start all blocks each time."""
    graph, queries, heavy, light = _mixed_graph()
    eng = E.Engine(graph, queries, relabel=False)
    try:
        first = _waves(eng, heavy)
        for _ in range(3):
            for _ in range(8):
                eng.process_batch(*light)
            assert _waves(eng, heavy) == first
    finally:
        eng.close()


def test_a_heavy_round_after_many_light_ones_is_joined_by_the_reserve():
    """Once light rounds have settled on few blocks, a heavy one gets as many again while it
    runs, and counts what it did; the light ones do without them."""
    graph, queries, heavy, light = _mixed_graph()
    eng = E.Engine(graph, queries, relabel=False)
    try:
        want = eng.process_batch(*heavy)[0].tolist()
        most = _waves(eng, heavy)
        for _ in range(400):
            eng.process_batch(*light)
        few = _waves(eng, light)
        assert 2 * few <= most
        assert eng.process_batch(*heavy)[0].tolist() == want and want[0] > 0
        s = eng.stats()
        assert s["dfs_waves"] // s["dfs_launches"] == 2 * few
    finally:
        eng.close()


@pytest.mark.parametrize("queue_capacity", [0, 1, 2, 50, 100000])
def test_few_hand_offs_are_allowed(queue_capacity):
    """A limit on a round's hand-offs below the number of its waves allows some: 400
    records of 200-entry lists, eight seeds each, more than the grid has waves."""
    n, rng = 2000, np.random.default_rng(9)
    i = np.arange(n)
    u = np.repeat(i, 100)
    v = (u + np.tile(rng.choice(np.arange(1, n // 2), 100, replace=False), n)) % n
    u, v, lab = u.astype(np.uint32), v.astype(np.uint32), np.zeros(n, np.uint32)
    sq = np.array([(0, 1), (1, 2), (2, 3), (3, 0)], np.uint32)
    queries = [(4, np.zeros(4, np.uint32), sq[:, 0].copy(), sq[:, 1].copy())]
    pick = rng.choice(len(u), 400, replace=False)
    batch = (np.ones(400, np.uint8), u[pick], v[pick], np.zeros(400, np.uint32))
    want = O.run_stream(O.Graph(n, lab, u, v), [O.Query(*queries[0])], [batch], relabel=False)[0]["pos"]
    eng = E.Engine((n, lab, u, v), queries, relabel=False, queue_capacity=queue_capacity)
    try:
        for _ in range(3):
            assert eng.process_batch(*batch)[0].tolist() == want
            donated = eng.stats()["tasks_donated"]
            assert (donated > 0) == (queue_capacity != 1)
            assert queue_capacity == 0 or donated < queue_capacity
    finally:
        eng.close()


@pytest.mark.parametrize("k,whole", [(4, False), (6, True), (9, True)])
def test_deep_queries_over_short_lists_get_a_block_per_cu(k, whole):
    """One record of a graph whose lists have 8 or 16 entries: a path of many vertices gives
    a whole grid work, one of four does not."""
    n, half, rng = 3000, 8 if k < 9 else 4, np.random.default_rng(k)
    i = np.arange(n)
    u = np.repeat(i, half).astype(np.uint32)
    v = ((u + np.tile(rng.choice(np.arange(1, n // 2), half, replace=False), n)) % n).astype(np.uint32)
    graph = (n, np.zeros(n, np.uint32), u, v)
    queries = [(k, np.zeros(k, np.uint32), np.arange(k - 1, dtype=np.uint32), np.arange(1, k, dtype=np.uint32))]
    one = (np.ones(1, np.uint8), u[:1], v[:1], np.zeros(1, np.uint32))
    full = (np.ones(2000, np.uint8), u[:2000], v[:2000], np.zeros(2000, np.uint32))
    eng = E.Engine(graph, [(2, np.zeros(2, np.uint32), np.zeros(1, np.uint32), np.ones(1, np.uint32))], relabel=False,
                   blocks_per_cu=1)
    try:
        grid = _waves(eng, full)  # a block per CU
    finally:
        eng.close()
    want = O.run_stream(O.Graph(*graph), [O.Query(*queries[0])], [one], relabel=False)[0]["pos"]
    eng = E.Engine(graph, queries, relabel=False)
    try:
        assert eng.process_batch(*one)[0].tolist() == want and want[0] > 0
        waves = _waves(eng, one)
        assert waves >= grid if whole else waves < grid
    finally:
        eng.close()
