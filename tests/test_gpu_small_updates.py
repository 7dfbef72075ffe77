"""Updates that one block applies, and their neighbours that many do: numbers of
touched lists, list lengths around the label-sorted copies and the pieces, relabels,
and a pool that has to grow in the middle."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TRI = np.array([(0, 1), (1, 2), (0, 2)], np.uint32)
QUERIES = [(3, np.array([0, 1, 2], np.uint32), TRI[:, 0].copy(), TRI[:, 1].copy()),
           (3, np.array([0, 0, 1], np.uint32), np.array([0, 1], np.uint32), np.array([1, 2], np.uint32))]


@pytest.mark.parametrize("records", [1, 2, 7, 16, 17, 40])
@pytest.mark.parametrize("hub", [3, 62, 64, 200, 1015, 1030])
@pytest.mark.parametrize("n", [1100, 65536, 65537])
@pytest.mark.parametrize("relabel", [True, False])
def test_small_updates(records, hub, n, relabel):
    rng = np.random.default_rng([records, hub, n])
    lab = rng.integers(0, 4, n).astype(np.uint32)
    u = np.concatenate([np.zeros(hub, np.uint32), rng.integers(1, 1100, 1500).astype(np.uint32)])
    v = np.concatenate([np.arange(1, hub + 1, dtype=np.uint32), rng.integers(1, 1100, 1500).astype(np.uint32)])
    keep = u != v
    u, v = u[keep], v[keep]
    batches = []
    for i in range(8):
        add = np.full(records, i % 2, np.uint8) if i < 4 else rng.integers(0, 2, records).astype(np.uint8)
        src, dst = rng.integers(0, 1090, records).astype(np.uint32), rng.integers(1090, 1100, records).astype(np.uint32)
        pick = rng.integers(0, len(u), records)
        gone = add == 0  # deletes of edges that are there, mostly
        src[gone], dst[gone] = u[pick][gone], v[pick][gone]
        src[0], dst[0] = 0, 1095 - i  # the hub's list in every batch
        batches.append((add, src, dst, rng.integers(0, 4, records).astype(np.uint32)))
    want = O.run_stream(O.Graph(n, lab, u, v), [O.Query(*q) for q in QUERIES], batches, relabel=relabel)
    g = O.Graph(n, lab, u, v)
    O.run_stream(g, [O.Query(*QUERIES[0])], batches, relabel=relabel)
    off, nb, dl = g.export()
    cand = g.candidates(O.Query(*QUERIES[0]))
    dl = np.where(dl == 3, 255, dl)  # a label no query uses
    for kw in (dict(), dict(overlap_apply=False)):
        eng = E.Engine((n, lab, u, v), QUERIES, relabel=relabel, **kw)
        try:
            for i, b in enumerate(batches):
                pos, neg = eng.process_batch(*b)
                assert pos.tolist() == want[i]["pos"] and neg.tolist() == want[i]["neg"], (kw, i)
            o2, n2, l2 = eng.graph()
            assert np.array_equal(off, o2) and np.array_equal(nb, n2) and np.array_equal(dl, l2)
            for q in range(3):
                assert np.array_equal(eng.candidates(0, q), cand[q].astype(bool)), q
        finally:
            eng.close()


@pytest.mark.parametrize("deletes", [0, 1])
def test_the_pool_grows_in_a_small_update(deletes):
    """4,000 lists of 700 entries filled to the end of their slots (879) by one batch,
    then moved to larger ones up to 32 a batch until there is no room for them; with a
    delete in every batch its round runs beside the update, ahead of the inserts'."""
    n = 4000
    i = np.arange(n)
    ring = [(i, (i + k) % n) for k in range(1, 351)]
    fill = [(i, (i + k) % n) for k in range(351, 440)] + [(i[:2000], i[:2000] + 2000)]
    over = (i[:2000], i[:2000] + 1000)

    def flat(edges):
        return (np.concatenate([e[0] for e in edges]).astype(np.uint32),
                np.concatenate([e[1] for e in edges]).astype(np.uint32))

    eng = E.Engine((n, np.zeros(n, np.uint32), *flat(ring)),
                   [(2, np.zeros(2, np.uint32), np.zeros(1, np.uint32), np.ones(1, np.uint32))])
    try:
        src, dst = flat(fill)
        pos, _ = eng.process_batch(np.ones(len(src), np.uint8), src, dst, np.zeros(len(src), np.uint32))
        assert pos.tolist() == [2 * len(src)]
        before = eng.stats()["pool_entries_capacity"]
        src, dst = flat([over])
        for x in range(0, 2000, 16):
            add = np.concatenate([np.ones(16, np.uint8), np.zeros(deletes, np.uint8)])
            gone = np.full(deletes, 3000 + x // 16 * 4, np.uint32)
            pos, neg = eng.process_batch(add, np.concatenate([src[x:x + 16], gone]),
                                         np.concatenate([dst[x:x + 16], gone + 5]), np.zeros(16 + deletes, np.uint32))
            assert pos.tolist() == [32] and neg.tolist() == [2 * deletes], x
        assert eng.stats()["pool_entries_capacity"] > before
        off, nb, _ = eng.graph()
    finally:
        eng.close()
    a, b = (x.astype(np.int64) for x in flat(ring + fill + [over]))
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    gone = np.arange(3000, 3500, 4) if deletes else np.zeros(0, np.int64)
    key = np.setdiff1d(key, np.concatenate([gone * n + gone + 5, (gone + 5) * n + gone]))
    assert np.array_equal(nb, (key % n).astype(np.uint32))
    assert np.array_equal(np.diff(off).astype(np.int64), np.bincount(key // n, minlength=n))
