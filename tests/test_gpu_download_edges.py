"""Labels to host memory at the exact sizes where the way there changes: one
piece up to half a MiB, pieces up to 8 MiB, one plain copy beyond; the last
piece whole, short by one element and of one or two elements."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

CHUNK = (1 << 19) // 4  # labels in a piece
MOST = 16 * CHUNK       # labels that go in pieces

# (points, variants)
SHAPES = [(CHUNK - 1, 1), (CHUNK, 1), (CHUNK + 1, 1), (2 * CHUNK - 1, 1), (3 * CHUNK + 2, 1),
          (MOST // 8 - 1, 8), (MOST // 8, 8), (MOST // 8 + 1, 8), (MOST - 1, 1), (MOST + 1, 1)]


@pytest.mark.parametrize("n,nvar", SHAPES)
def test_host_labels(n, nvar):
    words = n * nvar
    assert words in (CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK - 1, 3 * CHUNK + 2, MOST - 8, MOST,
                     MOST + 8, MOST - 1, MOST + 1)
    side = np.sqrt(n / 5.0)
    r = np.random.Generator(np.random.PCG64(words))
    x, y = r.uniform(0, side, n), r.uniform(0, side, n)
    mp = np.arange(2, 2 + nvar, dtype=np.uint32)
    print(n, "points x", nvar, "variants", flush=True)
    got = vd.cluster(x, y, np.full(nvar, 0.45), mp)
    want = oracle.libvdbscan(x, y, np.full(nvar, 0.45), mp)
    assert (got == want).all()
