"""Both intersection entry points at the sizes where a call takes another path: one
block for short first sets, one copy for short inputs and for short results."""
import numpy as np
import pytest

from dsm_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(1, 1), (1, 9000), (63, 64), (64, 65), (1024, 1025), (2047, 6145), (2048, 6144),
                                   (2048, 6145), (2049, 6143), (2049, 6144), (8192, 8192), (8193, 8192), (8193, 8193),
                                   (70000, 2), (65536 + 1, 65536 + 1)])
@pytest.mark.parametrize("spread", [1, 3])
@pytest.mark.parametrize("noalloc", [False, True])
def test_intersection_where_the_path_changes(na, nb, spread, noalloc):
    rng = np.random.default_rng([na, nb, spread])
    hi = spread * max(na, nb)
    a, b = (np.sort(rng.choice(hi, k, replace=False)).astype(np.uint32) for k in (na, nb))
    a[-1] = b[-1] = 0xFFFFFFFE  # the largest value
    assert np.array_equal(E.intersect_sorted(a, b, noalloc=noalloc), np.intersect1d(a, b))


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("na,nb,at", [(10, 9000, 8999), (10, 9000, 4500), (9000, 10, 0), (9000, 10, 8998),
                                      (9000, 9000, 255), (70000, 5, 69999), (5, 70000, 0)])
def test_long_inputs_out_of_order_are_refused(na, nb, at, noalloc):
    a, b = (np.arange(0, 2 * k, 2, dtype=np.uint32) for k in (na, nb))
    long = a if na >= nb else b
    for bad in (0xFFFFFFFF, long[at - 1] if at else long[1] + 5):
        keep, long[at] = long[at], bad
        with pytest.raises(E.DsmError) as ei:
            E.intersect_sorted(a, b, noalloc=noalloc)
        assert ei.value.code == E.DSM_EINVAL
        long[at] = keep
    assert np.array_equal(E.intersect_sorted(a, b, noalloc=noalloc), np.intersect1d(a, b))
