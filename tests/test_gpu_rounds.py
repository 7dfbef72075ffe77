"""How a DFS round spreads its work: seeds cut into shares, hand-offs between
waves and the end of the launch, at the grid's edges."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = {"edge": [(0, 1)], "path3": [(0, 1), (1, 2)], "tri_pendant": [(0, 1), (1, 2), (0, 2), (1, 3)],
          "house": [(0, 1), (1, 2), (2, 3), (3, 0), (0, 4), (1, 4)]}


def one_label(shape):
    e = np.array(SHAPES[shape], np.uint32)
    n = int(e.max()) + 1
    return n, np.zeros(n, np.uint32), e[:, 0].copy(), e[:, 1].copy()


@pytest.mark.parametrize("records", [1, 2, 127, 128, 129, 512, 513, 1025])
@pytest.mark.parametrize("queue_capacity", [0, 1])
def test_seed_shares_around_the_grid_size(records, queue_capacity):
    """One record to one per wave and beyond (a query edge gives two seeds per
    record, a path four, ...: 1,024 waves are met from both sides), with and
    without hand-offs, for queries of two vertices (a share holds a whole
    match) to five."""
    rng = np.random.default_rng(records)
    n, m = 150, 900
    key = rng.permutation(n * n)
    key = key[key // n < key % n][:m]
    u, v = (key // n).astype(np.uint32), (key % n).astype(np.uint32)
    queries = [one_label(s) for s in sorted(SHAPES)]
    labels = np.zeros(n, np.uint32)
    # re-inserted present edges: each seeds, and the graph stays as it is
    pick = rng.integers(0, len(u), records)
    z = np.zeros(records, np.uint32)
    batch = (np.ones(records, np.uint8), u[pick], v[pick], z)
    want = O.run_stream(O.Graph(n, labels, u, v), [O.Query(*q) for q in queries], [batch], relabel=False)[0]
    eng = E.Engine((n, labels, u, v), queries, relabel=False, queue_capacity=queue_capacity)
    try:
        for _ in range(3):  # the mailboxes are used again by every round
            pos, neg = eng.process_batch(*batch)
            assert pos.tolist() == want["pos"] and neg.tolist() == want["neg"]
        if queue_capacity:
            assert eng.stats()["tasks_donated"] == 0
    finally:
        eng.close()


def test_watchdog_ends_a_round_whose_waves_wait():
    """A round that keeps some waves waiting past watchdog_ms (long shares of
    one seed, hand-offs off) ends by itself with DSM_EDEVICE."""
    n = 300
    u, v = np.triu_indices(n, 1)
    u, v = u.astype(np.uint32), v.astype(np.uint32)
    eng = E.Engine((n, np.zeros(n, np.uint32), u, v), [one_label("house")], relabel=False, queue_capacity=1,
                   watchdog_ms=1, leaf_sets=False)
    try:
        with pytest.raises(E.DsmError) as ei:
            eng.process_batch(np.ones(1, np.uint8), u[:1], v[:1], np.zeros(1, np.uint32))
        assert ei.value.code == E.DSM_EDEVICE and "watchdog" in str(ei.value)
    finally:
        eng.close()


@pytest.mark.parametrize("da,db", [(5, 5000), (70, 20000), (128, 300), (129, 700), (130, 131), (900, 40000),
                                   (1024, 1500), (1025, 1026), (1026, 2047), (2048, 2049), (2050, 2051)])
@pytest.mark.parametrize("labels", [1, 2])
def test_leaf_sets_at_their_limits(da, db, labels):
    """Squares between two hubs of da and db neighbours: leaf sets of up to and
    past 128 entries (hash set or id ranges), 1,024 (kept or descended) and lists
    past 2,048 entries; lists short and long enough that the set's elements are
    searched in them; with the leaf's label that of other positions or not."""
    rng = np.random.default_rng(da + db)
    n = max(da, db) + 2
    xs = np.arange(2, n, dtype=np.uint32)
    pa, pb = rng.choice(xs, da, replace=False), rng.choice(xs, db, replace=False)
    extra = rng.choice(xs, (400, 2))
    u = np.concatenate([np.zeros(da, np.uint32), np.ones(db, np.uint32), extra[:, 0]]).astype(np.uint32)
    v = np.concatenate([pa, pb, extra[:, 1]]).astype(np.uint32)
    keep = u != v
    u, v = u[keep], v[keep]
    lab = np.zeros(n, np.uint32)
    lab[2:] = labels - 1
    sq = np.array([(0, 1), (1, 2), (2, 3), (3, 0)], np.uint32)
    queries = [(4, np.array([0, labels - 1] * 2, np.uint32), sq[:, 0].copy(), sq[:, 1].copy())]
    both = np.intersect1d(pa, pb)
    x = (both if len(both) else pa)[:2].astype(np.uint32)
    batch = (np.ones(4, np.uint8), np.array([0, 0, 1, 1], np.uint32),
             np.resize(x, 4).astype(np.uint32), np.zeros(4, np.uint32))
    want = O.run_stream(O.Graph(n, lab, u, v), [O.Query(*q) for q in queries], [batch], relabel=False)[0]
    for kw in ({}, {"leaf_segments": False}, {"leaf_budget": 64}):
        eng = E.Engine((n, lab, u, v), queries, relabel=False, **kw)
        try:
            pos, neg = eng.process_batch(*batch)
            assert pos.tolist() == want["pos"] and neg.tolist() == want["neg"], kw
        finally:
            eng.close()


@pytest.mark.parametrize("limit", [64, 1024, 2048, 4096, 8192, 65536, 524288])
def test_lists_that_grow_past_a_kernel_limit(limit):
    """A hub's list grows by one entry at a time from just below a length at which
    an update needs one more kernel to just above it, and shrinks again, one batch
    per call and pipelined: counts, graph and candidate bitmaps against the oracle."""
    n = limit + 40
    rng = np.random.default_rng(limit)
    lab = rng.integers(0, 3, n).astype(np.uint32)
    k = limit - 2
    u = np.concatenate([np.zeros(k, np.uint32), rng.integers(1, n, 300).astype(np.uint32)])
    v = np.concatenate([np.arange(1, k + 1, dtype=np.uint32), rng.integers(1, n, 300).astype(np.uint32)])
    keep = u != v
    u, v = u[keep], v[keep]
    tri = np.array([(0, 1), (1, 2), (0, 2)], np.uint32)
    queries = [(3, np.array([0, 1, 2], np.uint32), tri[:, 0].copy(), tri[:, 1].copy()), one_label("path3")]
    new = np.arange(k + 1, k + 7, dtype=np.uint32)
    batches = [(np.ones(1, np.uint8), np.zeros(1, np.uint32), x[None], lab[x][None]) for x in new]
    # delete one and insert one (the hub changes its label), so that the update runs beside a round
    batches += [(np.array([0, 1], np.uint8), np.array([0, x], np.uint32), np.array([x, x + 9], np.uint32),
                 np.full(2, (b + 1) % 3, np.uint32)) for b, x in enumerate(new[:3])]
    batches += [(np.array([1, 0], np.uint8), np.array([0, 0], np.uint32), np.array([x, x + 3], np.uint32),
                 np.full(2, b, np.uint32)) for b, x in enumerate(new[:3])]
    want = O.run_stream(O.Graph(n, lab, u, v), [O.Query(*q) for q in queries], batches)
    one, many = (E.Engine((n, lab, u, v), queries) for _ in range(2))
    try:
        pos, neg, _ = many.process_batches(batches)
        for i, b in enumerate(batches):
            p, m = one.process_batch(*b)
            assert p.tolist() == want[i]["pos"] == pos[i].tolist() and m.tolist() == want[i]["neg"] == neg[i].tolist(), i
        g = O.Graph(n, lab, u, v)
        O.run_stream(g, [O.Query(*queries[0])], batches)
        off, nb, dl = g.export()
        cand = g.candidates(O.Query(*queries[0]))
        for eng in (one, many):
            o2, n2, l2 = eng.graph()
            assert np.array_equal(off, o2) and np.array_equal(nb, n2) and np.array_equal(dl, l2)
            for q in range(3):
                assert np.array_equal(eng.candidates(0, q), cand[q].astype(bool)), q
    finally:
        one.close()
        many.close()


@pytest.mark.parametrize("n", [2, 3, 65, 2048, 2049, 70000])
@pytest.mark.parametrize("records", [255, 256, 2500])
def test_update_rule_on_conflicting_batches(n, records):
    """Batches just below and above the length sorted by counting passes, full of
    repeated and contradicting records of the same edges in both directions: the
    graph and labels after the update rule equal the oracle's."""
    rng = np.random.default_rng(n * 7 + records)
    lab = rng.integers(0, 4, n).astype(np.uint32)
    u, v = np.zeros(1, np.uint32), np.ones(1, np.uint32)
    pairs = rng.integers(0, n, (max(1, records // 6), 2)).astype(np.uint32)
    pairs[pairs[:, 0] == pairs[:, 1], 1] = 0
    pairs = pairs[pairs[:, 0] != pairs[:, 1]]
    if not len(pairs):
        pairs = np.array([[0, 1]], np.uint32)
    queries = [one_label("path3"), (2, np.array([1, 2], np.uint32), np.zeros(1, np.uint32), np.ones(1, np.uint32))]
    g = O.Graph(n, lab, u, v)
    eng = E.Engine((n, lab, u, v), queries)
    try:
        for _ in range(2):
            p = pairs[rng.integers(0, len(pairs), records)]
            turn = rng.random(records) < 0.5
            b = ((rng.random(records) < 0.6).astype(np.uint8), np.where(turn, p[:, 1], p[:, 0]),
                 np.where(turn, p[:, 0], p[:, 1]), rng.integers(0, 4, records).astype(np.uint32))
            O.run_stream(g, [], [b])
            eng.process_batch(*b)
            off, nb, dl = g.export()
            o2, n2, l2 = eng.graph()
            assert np.array_equal(off, o2) and np.array_equal(nb, n2)
            assert np.array_equal(np.where(dl > 2, 255, dl), l2)
    finally:
        eng.close()


def test_grids_follow_the_work_of_earlier_rounds():
    """Rounds of little work after a first one of unknown work start fewer blocks, and
    batches of other sizes in between change the grid again: counts against the oracle."""
    rng = np.random.default_rng(11)
    n, m = 4000, 60000
    u, v = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    keep = u != v
    u, v = u[keep], v[keep]
    lab = rng.integers(0, 2, n).astype(np.uint32)
    queries = [one_label("tri_pendant"), (3, np.array([0, 1, 0], np.uint32), np.array([0, 1], np.uint32),
                                          np.array([1, 2], np.uint32))]
    batches = []
    for k in (400, 1, 400, 400, 3000, 2, 50, 6000, 400):
        src, dst = rng.integers(0, n, k).astype(np.uint32), rng.integers(0, n, k).astype(np.uint32)
        batches.append((rng.integers(0, 2, k).astype(np.uint8), src, dst, lab[dst]))
    want = O.run_stream(O.Graph(n, lab, u, v), [O.Query(*q) for q in queries], batches)
    eng = E.Engine((n, lab, u, v), queries)
    try:
        waves = []
        for i, b in enumerate(batches):
            pos, neg = eng.process_batch(*b)
            assert pos.tolist() == want[i]["pos"] and neg.tolist() == want[i]["neg"], i
            s = eng.stats()
            waves.append(s["dfs_waves"] // s["dfs_launches"])
        assert waves[3] < waves[0]
    finally:
        eng.close()
