"""The cluster refinement of updates whose pool has to grow in the middle: lists have
moved then whose label-sorted copies are built only after the growth."""
import numpy as np
import pytest

from dsm_amd import engine as E
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DENSE, SPARSE = 4000, 600
QUERIES = [(3, np.array(lab, np.uint32), np.array(src, np.uint32), np.array(dst, np.uint32))
           for lab, src, dst in (([0, 1, 2], [0, 1, 0], [1, 2, 2]), ([1, 0, 1], [0, 1], [1, 2]))]


def flat(edges):
    return (np.concatenate([e[0] for e in edges]).astype(np.uint32),
            np.concatenate([e[1] for e in edges]).astype(np.uint32))


# inserts a batch once the pool is nearly full, and deletes, whose round runs beside the
# update (ahead of it, where one block applies it)
@pytest.mark.parametrize("records,deletes", [(16, 0), (15, 1), (400, 0), (400, 3)],
                         ids=["one block", "one block after a round", "in place", "overlapped"])
def test_refinement_of_an_update_that_grows_the_pool(records, deletes):
    """4,000 lists of 700 entries filled to the end of their slots (879) by one batch;
    the next moves 2,400 of them to slots of 1,108, which leaves room in the pool for 134
    more, and the batches after it move more than that. 600 short lists beside them, from
    which the refinement takes candidates. Updates of 16 records (32 lists) are applied by
    one block."""
    rng = np.random.default_rng(records + deletes)
    n = DENSE + SPARSE
    i = np.arange(DENSE)
    ring = [(i, (i + k) % DENSE) for k in range(1, 351)]
    fill = flat([(i, (i + k) % DENSE) for k in range(351, 440)] + [(i[:2000], i[:2000] + 2000)])
    thin = rng.integers(DENSE, n, (2, 900))
    thin = thin[:, thin[0] != thin[1]]
    lab = rng.integers(0, 4, n).astype(np.uint32)
    u, v = flat(ring + [(thin[0], thin[1])])
    g = O.Graph(n, lab, u, v)
    oq = [O.Query(*q) for q in QUERIES]
    batches = [(fill[0], fill[1], 0), (i[:1200], i[:1200] + 2001, 0)]
    batches += [(i[x:x + records], (i[x:x + records] + 2001) % DENSE, deletes)
                for x in range(1200, min(1200 + 6 * records, 2000), records)]
    batches.append((i[:records], i[:records] + 1300, deletes))
    eng = E.Engine((n, lab, u, v), QUERIES, relabel=False, cluster_filter=True)
    try:
        room, grown = eng.stats()["pool_entries_capacity"], []
        for b, (src, dst, gone) in enumerate(batches):
            out = 3000 + 7 * (b * deletes + np.arange(gone))  # edges of the ring
            batch = (np.r_[np.ones(len(src), np.uint8), np.zeros(gone, np.uint8)], np.r_[src, out].astype(np.uint32),
                     np.r_[dst, out + 5].astype(np.uint32), np.zeros(len(src) + gone, np.uint32))
            eng.apply_batch(*batch)
            if b == 0:  # too many records to count
                g.apply(*batch, relabel=False)
            else:
                want = O.run_stream(g, oq, [batch], relabel=False)[0]
                pos, neg = eng.match_batch()
                assert pos.tolist() == want["pos"] and neg.tolist() == want["neg"], b
            for q in range(len(QUERIES)):
                cand = g.cluster_candidates(oq[q])
                assert cand.any(1).all() and not cand.any(0).all()
                for x in range(3):
                    assert np.array_equal(eng.refined_candidates(q, x), cand[x].astype(bool)), (b, q, x)
            now = eng.stats()["pool_entries_capacity"]
            if b and now > room:
                grown.append(b)
            room = now
        # in the middle of the last kind of batches, with batches after it
        assert grown and 2 <= grown[0] < len(batches) - 1
        off, nb, _ = g.export()
        o2, n2, _ = eng.graph()
        assert np.array_equal(off, o2) and np.array_equal(nb, n2)
    finally:
        eng.close()
