"""Point order at the edges of the radix sort's tile sizes (1,024 items up to
65,536 points, 2,048 up to 131,072, 4,096 with offsets from the tiles' own
histograms up to 262,144 and from a scan beyond) and of the one-block scan
(16,384 elements): equal to the oracle's."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["spread", "one bin"])
@pytest.mark.parametrize("n", [16385, 17407, 17409, 65535, 65536, 65537, 67585, 131072, 131073,
                               262143, 262144, 262145, 266241])
def test_rank_order(n, kind):
    r = np.random.Generator(np.random.PCG64(n))
    if kind == "spread":
        x, y = r.uniform(-90, 90, n), r.uniform(-180, 180, n)
    else:  # nearly all points share a bin; order is the caller's
        x, y = r.uniform(10, 10.01, n), r.uniform(10, 10.01, n)
        x[-1], y[-1] = 80.0, 80.0
    print(n, kind, flush=True)
    assert (vd.rank_order(x, y) == oracle.bin_order(x, y)).all()


@pytest.mark.parametrize("n", [16385, 65537, 131073])
def test_labels(n):
    r = np.random.Generator(np.random.PCG64(n))
    x, y = r.uniform(0, 60, n), r.uniform(0, 60, n)
    for path in (vd.PATH_BATCH, vd.PATH_FUSED):
        got = vd.cluster(x, y, 0.2, 4, path=path)[0]
        assert (got == oracle.libvdbscan(x, y, [0.2], [4])[0]).all(), path
