"""Labels to host memory around the sizes at which the way there changes: up to
half a MiB in one piece, up to 8 MiB in pieces, beyond by one plain copy; the
last piece whole, of one element and short by one."""
import numpy as np
import pytest

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

CHUNK = (1 << 19) // 4


@pytest.mark.parametrize("words", [CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK - 1, 3 * CHUNK + 2,
                                   16 * CHUNK - 8, 16 * CHUNK, 16 * CHUNK + 8])
def test_host_labels_equal_device_order(words):
    # as many variants of one eps as make the array `words` long or just over
    n = 16_900
    r = np.random.Generator(np.random.PCG64(5))
    x, y = r.uniform(0, 30, n), r.uniform(0, 30, n)
    nvar = -(-words // n)
    n = words // nvar
    x, y = x[:n], y[:n]
    mp = np.arange(2, 2 + nvar, dtype=np.uint32) % 24 + 2
    print(n, "points x", nvar, "variants", flush=True)
    got = vd.cluster(x, y, np.full(nvar, 0.4), mp)
    one = {int(m): vd.cluster(x, y, 0.4, int(m))[0] for m in np.unique(mp)}
    for v in range(nvar):
        assert (got[v] == one[int(mp[v])]).all(), v
