"""The intersection entry points where their inputs stop going up in one copy (262,144
entries together, 131,072 without an allocation) and their results stop coming back in
one (at most half as many)."""
import numpy as np
import pytest

from dsm_amd import engine as E

pytestmark = pytest.mark.gpu

SIZES = [size for k in (65536, 131072)
         for size in ((k, k), (k - 1, k + 1), (k + 1, k - 1), (k, k + 1), (k + 1, k + 1), (2 * k - 1, 1), (2 * k, 1),
                      (1, 2 * k - 1), (1, 2 * k), (2048, 2 * k - 2048), (2048, 2 * k - 2047), (2049, 2 * k - 2049),
                      (2049, 2 * k - 2048), (300000, k))]


@pytest.mark.parametrize("na,nb", SIZES)
@pytest.mark.parametrize("noalloc", [False, True])
def test_intersection_around_the_staging_buffer(na, nb, noalloc):
    rng = np.random.default_rng([na, nb])
    a, b = (np.sort(rng.choice(2 * max(na, nb), k, replace=False)).astype(np.uint32) for k in (na, nb))
    a[-1] = b[-1] = 0xFFFFFFFE  # the largest value
    want = np.intersect1d(a, b)
    assert np.array_equal(E.intersect_sorted(a, b, noalloc=noalloc), want)
    # a call after one with bad inputs, and one of another size, finds nothing of theirs
    longer = a if na >= nb else b
    keep, longer[len(longer) // 2] = longer[len(longer) // 2], 0
    with pytest.raises(E.DsmError) as ei:
        E.intersect_sorted(a, b, noalloc=noalloc)
    assert ei.value.code == E.DSM_EINVAL
    longer[len(longer) // 2] = keep
    assert np.array_equal(E.intersect_sorted(a[:1], b[-1:], noalloc=noalloc), np.intersect1d(a[:1], b[-1:]))
    assert np.array_equal(E.intersect_sorted(a, b, noalloc=noalloc), want)
