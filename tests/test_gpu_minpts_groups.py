"""Batched engine around its groups of 8 minpts values: one, a full group, one
beyond it and two groups and one, with values that make every point core (1)
and none (above the point count), on points whose levels leave pairs open from
one level to the next; and cell pairs of few points around the sizes at which
they are looked at one by one. Labels are the oracle's."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd
from variantdbscan_amd import datasets

pytestmark = pytest.mark.gpu

N = 12_000
MINPTS = [1, 4, 2, 9, 6, 30, 3, 50_000, 5, 12, 7, 16, 8, 60, 25, 40, 100]


@pytest.fixture(scope="module")
def points():
    # filaments and noise beside a knot far denser than the rest
    x, y = datasets.aniso(N - 2000, seed=57)
    r = np.random.default_rng(58)
    kx, ky = r.normal(x.mean(), 0.15, 2000), r.normal(y.mean(), 0.15, 2000)
    return np.concatenate([x, kx]), np.concatenate([y, ky])


@pytest.mark.parametrize("levels", [1, 4], ids=["one-level", "four-levels"])
@pytest.mark.parametrize("nmp", [1, 7, 8, 9, 17])
def test_minpts_groups(points, nmp, levels):
    x, y = points
    E = [0.3, 0.37, 0.55, 0.8][:levels]
    eps = np.repeat(E, nmp)
    mp = np.tile(np.array(MINPTS[:nmp], dtype=np.uint32), levels)
    print("12k points, %d minpts values x %d levels" % (nmp, levels), flush=True)
    got = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH)
    want = oracle.libvdbscan(x, y, eps, mp)
    for v in range(len(eps)):
        assert (got[v] == want[v]).all(), (eps[v], mp[v])


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 9])
def test_cells_of_few_points(m):
    # tight knots of 1..m points on a jittered lattice of about eps spacing:
    # pairs of 1 x 1 up to m x m points, near the thresholds of every level
    r = np.random.default_rng(70 + m)
    gx, gy = np.meshgrid(np.arange(40) * 0.5, np.arange(37) * 0.5)
    cx = gx.ravel() + r.uniform(-0.06, 0.06, gx.size)
    cy = gy.ravel() + r.uniform(-0.06, 0.06, gy.size)
    rep = r.integers(1, m + 1, cx.size)
    x, y = np.repeat(cx, rep), np.repeat(cy, rep)
    x = x + r.uniform(-0.05, 0.05, x.size)
    y = y + r.uniform(-0.05, 0.05, y.size)
    eps = np.repeat([0.45, 0.5, 0.52, 0.6], 3)
    mp = np.tile(np.array([2, m + 2, 2 * m + 3], dtype=np.uint32), 4)
    print("knots of 1..%d points" % m, flush=True)
    got = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH)
    want = oracle.libvdbscan(x, y, eps, mp)
    for v in range(len(eps)):
        assert (got[v] == want[v]).all(), (eps[v], mp[v])


@pytest.mark.parametrize("border", [vd.BORDER_REFERENCE, vd.BORDER_STANDARD], ids=["ref", "std"])
@pytest.mark.parametrize("levels,nmp", [(1, 1), (1, 3), (1, 8), (2, 1), (4, 5), (7, 1), (15, 1),
                                        (15, 8), (16, 2)])
def test_label_shapes(points, levels, nmp, border):
    # level and minpts counts on both sides of every shape of the label pass
    x, y = points[0][::4], points[1][::4]
    E = np.round(np.linspace(0.3, 1.1, levels), 4)
    M = np.array([4, 6, 9, 12, 3, 20, 7, 2], dtype=np.uint32)[:nmp]
    eps, mp = np.repeat(E, nmp), np.tile(M, levels)
    keep = np.arange(len(eps)) % 5 != 3  # some (level, value) pairs not asked for
    eps, mp = eps[keep], mp[keep]
    print("%d levels x %d minpts values" % (levels, nmp), flush=True)
    got = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH, border=border)
    if border == vd.BORDER_REFERENCE:
        want = oracle.libvdbscan(x, y, eps, mp)
    else:
        from sklearn.cluster import DBSCAN
        X = np.column_stack([x, y])
        want = [DBSCAN(eps=e, min_samples=int(m), algorithm="kd_tree").fit(X).labels_
                for e, m in zip(eps, mp)]
    for v in range(len(eps)):
        assert (got[v] == want[v]).all(), (eps[v], mp[v])
