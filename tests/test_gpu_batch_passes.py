"""Batched engine: numbers of minpts values around the groups of 8 that run side
by side, values that every point and no point reaches, calls whose values run in
several passes (within a word of 8 levels, whole words, an odd rest), and lists
numbered before they are stored. Every variant runs batched; labels are the
oracle's, the standard rule's scikit-learn's."""
import numpy as np
import pytest
from sklearn.cluster import DBSCAN

import oracle

import variantdbscan_amd as vd
from variantdbscan_amd import _lib, datasets

pytestmark = pytest.mark.gpu

NONE = 0x80000000  # a minpts value that nothing reaches
MINPTS = [4, NONE, 2, 9, 6, 30, 3, 1, 5, 12, 7, 16, 8, 60, 25, 40, 33, 20]  # all different
E = [0.3, 0.37, 0.55, 0.8]


@pytest.fixture(scope="module")
def points():
    # filaments and noise beside a knot far denser than the rest
    x, y = datasets.aniso(9_000, seed=57)
    r = np.random.default_rng(58)
    kx, ky = r.normal(x.mean(), 0.15, 1_500), r.normal(y.mean(), 0.15, 1_500)
    return np.concatenate([x, kx]), np.concatenate([y, ky])


_want = {}


def _check(points, eps, mp, border=vd.BORDER_REFERENCE, tag=None):
    x, y = points
    got, st = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH, border=border, return_stats=True)
    info = _lib.batch_info()
    assert st["path_used"] == vd.PATH_BATCH
    assert info["minpts_values"] == len(set(mp)) and info["levels"] == len(set(eps))
    for v, (e, m) in enumerate(zip(eps, mp)):
        key = (tag, float(e), int(m), border)
        if key not in _want:
            if border == vd.BORDER_REFERENCE:
                _want[key] = oracle.libvdbscan(x, y, [e], [m])[0]
            else:
                _want[key] = DBSCAN(eps=e, min_samples=int(m), algorithm="kd_tree").fit(
                    np.column_stack([x, y])).labels_
        assert (got[v] == _want[key]).all(), (e, m)
    return info


def _cross(levels, values):
    return (np.repeat(levels, len(values)),
            np.tile(np.array(values, dtype=np.uint32), len(levels)))


@pytest.mark.parametrize("levels", [1, 4])
@pytest.mark.parametrize("nmp", [1, 7, 8, 9, 16, 17])
def test_groups(points, nmp, levels):
    eps, mp = _cross(E[:levels], MINPTS[:nmp])
    print(nmp, "minpts values x", levels, "levels", flush=True)
    _check(points, eps, mp)


@pytest.mark.parametrize("border", [vd.BORDER_REFERENCE, vd.BORDER_STANDARD], ids=["ref", "std"])
@pytest.mark.parametrize("nmp,most", [(3, 1), (7, 4), (8, 2), (9, 8), (12, 8), (13, 4), (17, 8),
                                      (17, 1), (17, 16)])
def test_passes(points, monkeypatch, nmp, most, border):
    # (the standard rule's reference refuses values beyond int32)
    values = [m for m in MINPTS if m != NONE or border == vd.BORDER_REFERENCE][:nmp]
    eps, mp = _cross(E[:3], values)
    keep = np.arange(len(eps)) % 7 != 5  # some pairs not asked for
    eps, mp = eps[keep], mp[keep]
    monkeypatch.setenv("VDB_BATCH_PASS_VALUES", str(most))
    for i in range(3):  # direct, captured, replayed
        print(len(values), "values, at most", most, "to a pass, call", i, flush=True)
        info = _check(points, eps, mp, border)
        # worklist totals are only kept where one pass takes all values
        assert info["fresh_pairs"] == 0
    monkeypatch.delenv("VDB_BATCH_PASS_VALUES")
    assert _check(points, eps, mp, border)["fresh_pairs"] > 0


@pytest.mark.parametrize("levels", [15, 16, 20])
def test_passes_of_many_levels(points, monkeypatch, levels):
    eps, mp = _cross(np.round(np.linspace(0.3, 0.9, levels), 4), MINPTS[:10])
    keep = np.arange(len(eps)) % 3 == 0
    monkeypatch.setenv("VDB_BATCH_PASS_VALUES", "4")
    print(levels, "levels, 10 values, 4 to a pass", flush=True)
    _check(points, eps[keep], mp[keep])


@pytest.mark.parametrize("border", [vd.BORDER_REFERENCE, vd.BORDER_STANDARD], ids=["ref", "std"])
@pytest.mark.parametrize("levels", [1, 4, 17])
def test_numbered_lists(points, monkeypatch, levels, border):
    eps, mp = _cross(np.round(np.linspace(0.3, 0.8, levels), 4), [4, 12, 9])
    monkeypatch.setenv("VDB_BATCH_LIST_BYTES", "1024")
    print("numbered lists,", levels, "levels", flush=True)
    info = _check(points, eps, mp, border)
    # the knot's cells hold more points than the longest list: none for those
    assert 0 < info["listed_points"] < len(points[0])


def test_numbered_lists_of_sets(points, monkeypatch):
    monkeypatch.setenv("VDB_BATCH_LIST_BYTES", "1024")
    sets = [points, (points[0][:700], points[1][:700]), (points[0][::3], points[1][::3])]
    got, st = vd.cluster_multi(sets, [0.3, 0.8], [4, 12], path=vd.PATH_BATCH, return_stats=True)
    assert st["path_used"] == vd.PATH_BATCH
    for g, s in zip(got, sets):
        assert (g == oracle.libvdbscan(s[0], s[1], [0.3, 0.8], [4, 12])).all()
