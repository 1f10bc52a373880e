"""Batched engine: the neighbour search by window population. Points of small
windows take a thread each, of middling ones 16 lanes, of crowded ones a wave,
and beyond 16 eps levels all take the wave; the sets here have windows on both
sides of every line (128 and 512 points), lists that fill up and shrink, and
window rows of strips one to four columns wide. Labels must equal the
oracle's bit for bit."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu


def _graded(seed, n=9000):
    """Density falling by a factor of about 2,000 from a clump to the edge."""
    r = np.random.Generator(np.random.PCG64(seed))
    rad = 12.0 * r.uniform(0.0, 1.0, n) ** 1.7
    t = r.uniform(0.0, 2.0 * np.pi, n)
    return rad * np.cos(t), rad * np.sin(t)


def _lattice(side, step):
    a = np.arange(side) * step
    return np.repeat(a, side), np.tile(a, side)


# (eps levels, smallest eps, largest eps, minpts values)
CASES = [(1, 0.4, 0.4, (5, 64)), (2, 0.2, 0.3, (2, 8, 33)), (4, 0.2, 0.8, (1, 4, 64)),
         (5, 0.25, 1.0, (3, 16, 40)), (8, 0.15, 0.9, (4, 8, 48)), (9, 0.1, 0.7, (5, 31)),
         (16, 0.1, 0.4, (6, 64)), (17, 0.1, 0.5, (6, 20)), (3, 0.05, 0.75, (4, 12))]


@pytest.mark.parametrize("case", CASES, ids=["K%d-%g-%g" % c[:3] for c in CASES])
def test_windows_of_every_population(case):
    K, lo, hi, minpts = case
    x, y = _graded(7 + K)
    E = np.round(np.linspace(lo, hi, K), 6)
    eps = np.repeat(E, len(minpts))
    mp = np.tile(np.array(minpts, dtype=np.uint32), K)
    print("graded 9,000 points, %d levels, batch" % K, flush=True)
    got, st = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH, return_stats=True)
    assert st["path_used"] == vd.PATH_BATCH
    want = oracle.libvdbscan(x, y, eps, mp)
    for v in range(len(eps)):
        assert (got[v] == want[v]).all(), (eps[v], mp[v])


@pytest.mark.parametrize("side,step", [(40, 0.25), (40, 0.1), (64, 0.0625)])
def test_lattice_at_spacing_multiples(side, step):
    """Distances equal to eps, many neighbours at one level."""
    x, y = _lattice(side, step)
    eps = np.repeat([step, 2 * step, 5 * step], 3)
    mp = np.tile(np.array([4, 5, 13], dtype=np.uint32), 3)
    got = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH)
    want = oracle.libvdbscan(x, y, eps, mp)
    assert (got == want).all()


def test_numbered_lists():
    """Above 8 GB of lists the listed points are numbered first."""
    n = 27_000_000
    r = np.random.Generator(np.random.PCG64(5))
    x, y = r.uniform(0.0, 300.0, n), r.uniform(0.0, 300.0, n)
    print("27M uniform points, minpts 64", flush=True)
    a = vd.cluster(x, y, 0.25, 64, path=vd.PATH_BATCH)
    b = vd.cluster(x, y, 0.25, 64, path=vd.PATH_FUSED, cells_per_eps=2)
    assert a.max() > 0
    assert (a == b).all()
    vd._lib.load().vdb_release()
