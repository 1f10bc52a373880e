"""Window rows from the bitset of occupied keys, and by search beyond its
limits (512 keys a cell or 2^25 keys): key spaces on both sides of both lines,
keys at the ends of words, several datasets. Labels and counts must equal the
oracle's."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu


def _pairs(n, span, eps, seed):
    """n/3 uniform points with two companions each within eps, the box's corners."""
    r = np.random.Generator(np.random.PCG64(seed))
    m = n // 3
    x, y = r.uniform(0, span, m), r.uniform(0, span, m)
    x = np.concatenate([x, x + 0.5 * eps, x - 0.3 * eps, [0.0, span]])
    y = np.concatenate([y, y - 0.4 * eps, y + 0.9 * eps, [0.0, span]])
    return np.clip(x, 0, span), np.clip(y, 0, span)


# cells across the box at one cell per eps; the grids have 1 to 4 times as many
@pytest.mark.parametrize("n,across", [(17_000, 31), (17_000, 32), (17_000, 33), (20_000, 1440),
                                      (20_000, 2900), (20_000, 4090), (90_000, 3300),
                                      (90_000, 4700), (90_000, 9000)])
def test_rows_over_key_spaces(n, across):
    eps = 64.0 / across
    x, y = _pairs(n, 64.0, eps, n + across)
    print("%d points, %d cells across" % (len(x), across), flush=True)
    want = oracle.libvdbscan(x, y, [eps], np.array([3], dtype=np.uint32))
    for path in (vd.PATH_BATCH, vd.PATH_FUSED):
        got = vd.cluster(x, y, [eps], [3], path=path)
        assert (np.asarray(got).reshape(-1) == np.asarray(want).reshape(-1)).all(), path


def test_rows_of_many_datasets():
    sets = [_pairs(n, 40.0, 40.0 / a, a) for n, a in ((5_000, 31), (23, 3000), (9_001, 2048),
                                                     (3, 1), (12_000, 700))]
    E, M = [40.0 / 2048, 40.0 / 700], [3, 4]
    got = vd.cluster_multi(sets, E, M)
    for (x, y), g in zip(sets, got):
        want = oracle.libvdbscan(x, y, E, np.array(M, dtype=np.uint32))
        assert (np.asarray(g) == want).all()
