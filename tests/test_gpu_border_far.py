"""Border pass of the per-variant engine where most points are not core: from
65,536 such points of crowded windows on, a wave takes two of a cell together,
from 262,144 on eight, and passes over stretches without a core point. Sets on
both sides of these lines, with no, few and many core points, under both border
rules."""
import numpy as np
import pytest
from sklearn.cluster import DBSCAN

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

EPS = 1.0


def _points(n):
    """About 140 neighbours each (windows of about 270 points), evenly strewn,
    so that a minpts near that splits them: at 80,000 points 73,382, 4,375, 45
    and no core points for the minpts below, 72,000 to 77,000 listed for the others."""
    side = np.sqrt(n * np.pi * EPS * EPS / 140.0)
    r = np.random.Generator(np.random.PCG64(n))
    return r.uniform(0.0, side, n), r.uniform(0.0, side, n)


@pytest.mark.parametrize("minpts", [120, 160, 180, 5000])
@pytest.mark.parametrize("n", [60_000, 80_000, 310_000])
def test_few_core_points(n, minpts):
    x, y = _points(n)
    print(n, "points, minpts", minpts, flush=True)
    got = vd.cluster(x, y, EPS, minpts, path=vd.PATH_FUSED)[0]
    assert (got == oracle.libvdbscan(x, y, [EPS], [minpts])[0]).all()


@pytest.mark.parametrize("minpts", [160, 180])
def test_few_core_points_standard_rule(minpts):
    x, y = _points(80_000)
    print("standard rule, minpts", minpts, flush=True)
    got = vd.cluster(x, y, EPS, minpts, path=vd.PATH_FUSED, border=vd.BORDER_STANDARD)[0]
    want = DBSCAN(eps=EPS, min_samples=minpts, algorithm="kd_tree").fit(np.column_stack([x, y]))
    assert (got == want.labels_).all()


def test_knots_of_few_points():
    """Eight at a time over cells of 1 to about 20 points, and a crowded knot."""
    r = np.random.Generator(np.random.PCG64(3))
    n = 130_000
    x, y = r.normal(0.0, 6.0, n), r.normal(0.0, 6.0, n)
    x[::97], y[::97] = r.uniform(0, 0.02, x[::97].size), r.uniform(0, 0.02, x[::97].size)
    mp = [1340, 1500]  # the knot is core, and little else
    print("130,000 normal points with a knot", flush=True)
    got = vd.cluster(x, y, [0.4, 0.4], mp, path=vd.PATH_FUSED)
    want = oracle.libvdbscan(x, y, [0.4, 0.4], mp)
    assert (got == want).all()
