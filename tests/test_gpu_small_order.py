"""Point and cell order at the edges of the sorts: one block for up to 16,384
points (4 rounds of 1,024 items up to 4,096, else 16), tiles of 4,096 items in
passes of 8 or 9 bits beyond. Orders and labels must equal the oracle's."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

SIZES = [2, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 5120, 9999, 16383, 16384, 16385,
         20480, 20481]


def _points(n, kind):
    r = np.random.Generator(np.random.PCG64(n))
    if kind == "spread":
        return r.uniform(-90, 90, n), r.uniform(-180, 180, n)
    if kind == "one bin":  # nearly all points share a bin; order is the caller's
        x, y = r.uniform(10, 10.01, n), r.uniform(10, 10.01, n)
        x[-1], y[-1] = 80.0, 80.0
        return x, y
    # repeated points on a lattice
    x, y = r.integers(0, 40, n).astype(np.float64), np.sort(r.integers(0, 40, n)).astype(np.float64)
    x[0], y[0], x[-1], y[-1] = 0.0, 0.0, 39.0, 39.0
    return x, y


@pytest.mark.parametrize("kind", ["spread", "one bin", "lattice"])
@pytest.mark.parametrize("n", SIZES)
def test_rank_order(n, kind):
    x, y = _points(n, kind)
    assert (vd.rank_order(x, y) == oracle.bin_order(x, y)).all()


# eps 3, 0.4 and 0.02: cell keys of about 15, 20 and 28 bits
@pytest.mark.parametrize("n", [65, 1025, 4097, 16384, 16385, 20481])
def test_labels_over_key_widths(n):
    x, y = _points(n, "spread")
    for eps in (3.0, 0.4, 0.02):
        for path in (vd.PATH_BATCH, vd.PATH_FUSED):
            got = vd.cluster(x, y, eps, 3, path=path)[0]
            assert (got == oracle.libvdbscan(x, y, [eps], [3])[0]).all(), (eps, path)


def test_non_finite_and_overflow_are_refused():
    x, y = _points(3000, "spread")
    for bad in (np.nan, np.inf, -np.inf):
        z = x.copy()
        z[1234] = bad
        with pytest.raises(vd._lib.VdbError, match="non-finite"):
            vd.cluster(z, y, 0.5, 4)
    z = x.copy()
    z[0], z[1] = -1.7e308, 1.7e308
    with pytest.raises(vd._lib.VdbError):
        vd.cluster(z, y, 0.5, 4)
    assert (vd.cluster(x, y, 0.5, 4) == oracle.libvdbscan(x, y, [0.5], [4])).all()
