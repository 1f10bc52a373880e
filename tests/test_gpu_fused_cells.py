"""Fused engine: counts that stop at minpts (a thread per point up to windows
of 192 points, a wave per 8 origins beyond), components over clique cells (or
over points where a cell is no clique: one cell per eps), and border points by
window population. Labels must equal the oracle's bit for bit."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu


def _graded(seed, n=7000):
    """Density falling by a factor of about 2,000 from a clump to the edge."""
    r = np.random.Generator(np.random.PCG64(seed))
    rad = 10.0 * r.uniform(0.0, 1.0, n) ** 1.7
    t = r.uniform(0.0, 2.0 * np.pi, n)
    return rad * np.cos(t), rad * np.sin(t)


@pytest.mark.parametrize("cells", [0, 1, 2, 3, 8])
@pytest.mark.parametrize("eps", [0.15, 0.6, 2.5])
def test_minpts_on_both_sides_of_every_window(eps, cells):
    x, y = _graded(int(eps * 100))
    mp = np.array([0, 1, 5, 65, 191, 192, 193, 400, 7000, 7001, 0x80000000], dtype=np.uint32)
    e = np.full(len(mp), eps)
    print("graded 7,000 points, eps %g, fused, cells %d" % (eps, cells), flush=True)
    got = vd.cluster(x, y, e, mp, path=vd.PATH_FUSED, cells_per_eps=cells)
    want = oracle.libvdbscan(x, y, e, mp)
    for v in range(len(mp)):
        assert (got[v] == want[v]).all(), int(mp[v])


@pytest.mark.parametrize("border", [vd.BORDER_REFERENCE, vd.BORDER_STANDARD], ids=["ref", "std"])
def test_one_minpts_at_a_time_and_the_table(border):
    """The largest minpts of an eps bounds its counts: alone, together with
    smaller ones and with the table's exact counts, the labels are the same."""
    x, y = _graded(3)
    mp = np.array([3, 70, 150, 300], dtype=np.uint32)
    e = np.full(len(mp), 0.8)
    together = vd.cluster(x, y, e, mp, path=vd.PATH_FUSED, border=border)
    table = vd.cluster(x, y, e, mp, path=vd.PATH_TABLE, border=border)
    assert (together == table).all()
    for v in range(len(mp)):
        alone = vd.cluster(x, y, e[v:v + 1], mp[v:v + 1], path=vd.PATH_FUSED, border=border)
        assert (alone[0] == together[v]).all(), int(mp[v])


@pytest.mark.parametrize("path", [vd.PATH_FUSED, vd.PATH_TABLE], ids=["fused", "table"])
def test_gaps_of_one_ulp_between_dense_cells(path):
    """Two dense columns whose nearest points are exactly eps, then just over
    eps, apart: every cell pair across the gap is tested to the end."""
    r = np.random.Generator(np.random.PCG64(9))
    ya, yb = r.uniform(0, 2, 3000), r.uniform(0, 2, 3000)
    for gap, joined in ((0.5, True), (np.nextafter(0.5, 1.0), False)):
        x = np.concatenate([-r.uniform(0, 0.3, 3000), gap + r.uniform(0, 0.3, 3000)])
        y = np.concatenate([ya, yb])
        x[0], x[3000] = 0.0, gap
        y[0] = y[3000] = 1.0
        got = vd.cluster(x, y, 0.5, 80, path=path)[0]
        assert (got == oracle.libvdbscan(x, y, [0.5], [80])[0]).all()
        assert (got[0] == got[3000]) == joined
