"""Core test of the per-variant engine: counts stop at the largest minpts value
of an eps and where the candidates left cannot bring a point to its next value.
Sets with windows below and above 192 points, values on both sides of the
counts, one to more than eight of them, zero and such as nothing reaches."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

VALUES = [[140], [193], [5000], [100, 140, 180], [3, 140, 5000], [0, 20, 150],
          [0x80000000], [150, 0x80000000, 0xffffffff],
          [10, 60, 110, 120, 130, 140, 150, 160],            # eight
          [10, 60, 110, 120, 130, 140, 150, 160, 170],       # nine: any count matters
          list(range(120, 170, 2)) + [20_000]]


@pytest.fixture(scope="module")
def points():
    # even ground of about 140 neighbours (windows of 270 points), thin ground
    # of about 30, and a knot in a single cell
    r = np.random.Generator(np.random.PCG64(11))
    side = np.sqrt(20_000 * np.pi / 140.0)
    x = [r.uniform(0, side, 20_000), r.uniform(side + 1, 2 * side + 1, 4_000),
         r.uniform(5.1, 5.2, 700)]
    y = [r.uniform(0, side, 20_000), r.uniform(0, side, 4_000), r.uniform(5.1, 5.2, 700)]
    p = r.permutation(24_700)
    return np.concatenate(x)[p], np.concatenate(y)[p]


@pytest.mark.parametrize("minpts", VALUES, ids=[str(i) for i in range(len(VALUES))])
def test_values_of_one_eps(points, minpts):
    x, y = points
    eps = [1.0] * len(minpts)
    print("minpts", minpts, flush=True)
    got = vd.cluster(x, y, eps, minpts, path=vd.PATH_FUSED)
    want = oracle.libvdbscan(x, y, eps, minpts)
    for v in range(len(eps)):
        assert (got[v] == want[v]).all(), minpts[v]


@pytest.mark.parametrize("k", [1, 3, 8])
def test_other_resolutions(points, k):
    x, y = points
    minpts = [30, 141, 160, 900]
    print(k, "cells per eps", flush=True)
    got = vd.cluster(x, y, [1.0] * 4, minpts, path=vd.PATH_FUSED, cells_per_eps=k)
    assert (got == oracle.libvdbscan(x, y, [1.0] * 4, minpts)).all()
