"""Graph replays when a later call leaves its cell order in another buffer.

The cell order ends in whichever of two buffers the sort's last pass wrote, so
it changes place where the number of passes does, at 2^18 grid keys. The sets
here differ only in how far out their one outlier lies: same point count, same
cells, same cell pairs, on the two sides of that line. Labels must be the
oracle's whichever of them was captured."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

EPS, MINPTS = [0.5, 0.5], [6, 9]


def _set(x_far):
    """20,000 points thin enough for many border points, and an outlier."""
    r = np.random.Generator(np.random.PCG64(17))
    x, y = r.uniform(20.0, 75.0, 19_998), r.uniform(20.0, 75.0, 19_998)
    # the corner points fix the grid's origin and its 513 rows
    return np.concatenate([[0.0, x_far], x]), np.concatenate([[0.0, 181.0], y])


def _cells(x_far):
    """Columns (to whole strips of two) times rows of the grid at EPS[0]."""
    d = EPS[0] / np.sqrt(2.0) * (1.0 - 2.0 ** -20)
    ncx, ncy = int(x_far // d) + 2, int(181.0 // d) + 2
    return (ncx + 1) // 2 * 2 * ncy


NEAR, FAR = 178.0, 185.0


@pytest.mark.parametrize("first,then", [(NEAR, FAR), (FAR, NEAR)], ids=["outward", "inward"])
def test_cell_order_in_the_other_buffer(first, then):
    assert _cells(NEAR) < 1 << 18 < _cells(FAR)
    a, b = _set(first), _set(then)
    vd.cluster(*b, EPS, MINPTS, path=vd.PATH_BATCH)  # no buffer grows later
    for i in range(4):  # direct, captured, replayed twice
        print("set A, call", i, flush=True)
        got, st = vd.cluster(*a, EPS, MINPTS, path=vd.PATH_BATCH, return_stats=True)
        info = vd._lib.batch_info()
    assert st["path_used"] == vd.PATH_BATCH
    assert (got == oracle.libvdbscan(*a, EPS, MINPTS)).all()
    want = oracle.libvdbscan(*b, EPS, MINPTS)
    for i in range(3):
        print("set B, call", i, flush=True)
        got = vd.cluster(*b, EPS, MINPTS, path=vd.PATH_BATCH)
        assert vd._lib.batch_info() == info  # the same cells and pairs
        assert (got == want).all(), i


def test_sets_of_one_call_in_the_other_buffer():
    # two datasets in a call, the second's outlier on either side in turn
    inner = 76.0
    small = _set(inner)
    near, far = 100.0, 108.0
    assert _cells(inner) + _cells(near) < 1 << 18 < _cells(inner) + _cells(far)
    for x_far in (far, near, far):
        b = _set(x_far)
        want = [oracle.libvdbscan(*s, EPS, MINPTS) for s in (small, b)]
        for i in range(4):
            print("outlier at", x_far, "call", i, flush=True)
            got, st = vd.cluster_multi([small, b], EPS, MINPTS, path=vd.PATH_BATCH,
                                       return_stats=True)
            assert st["path_used"] == vd.PATH_BATCH
            for g, w in zip(got, want):
                assert (g == w).all(), i
