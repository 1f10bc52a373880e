"""Points of small windows, taken by a thread each, beside those taken by waves:
knots whose windows hold just under, at and just over the limit between the two
(192 points), single points, and all of one kind. Counts, table rows, digests
and the table engine's labels against brute force and the oracle."""
import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd

pytestmark = pytest.mark.gpu

EPS = 0.5
KNOTS = {
    "limit": [191, 192, 193, 64, 1, 257],
    "few": [1, 2, 7, 8, 9, 190],
    "many": [193, 200, 333],
    "one-point": [1],
}


def _points(sizes, seed):
    r = np.random.default_rng(seed)
    xs, ys = [], []
    for k, m in enumerate(sizes * 5):
        # knots of radius about eps, far enough apart not to meet
        xs.append(8.0 * k + r.uniform(-0.4, 0.4, m))
        ys.append(3.0 * (k % 7) + r.uniform(-0.4, 0.4, m))
    x, y = np.concatenate(xs), np.concatenate(ys)
    p = r.permutation(len(x))
    return x[p], y[p]


def _within(x, y):
    # the distance as the library defines it: separately rounded squares
    dx, dy = x[:, None] - x[None, :], y[:, None] - y[None, :]
    s = dx * dx + dy * dy
    return s <= EPS * EPS, s


@pytest.mark.parametrize("prec", [vd.PREC_FP64, vd.PREC_FP32_RECHECK], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", sorted(KNOTS))
def test_few(name, prec):
    x, y = _points(KNOTS[name], 11)
    print(name, len(x), "points, precision", prec, flush=True)
    inside, s = _within(x, y)
    assert (vd.neighbor_counts(x, y, EPS, precision=prec) == inside.sum(1)).all()
    off, ids, d2 = vd.neighbor_table(x, y, EPS, with_d2=True, precision=prec)
    assert (np.diff(off.astype(np.int64)) == inside.sum(1)).all()
    for i in range(len(x)):
        row = ids[off[i]:off[i + 1]]
        o = np.argsort(row)
        assert (row[o] == np.nonzero(inside[i])[0]).all()
        assert (d2[off[i]:off[i + 1]][o] == s[i, row[o]].astype(np.float32)).all()
    off1, ids1, _ = vd.neighbor_table(x, y, EPS, precision=prec)
    assert (off1 == off).all() and (ids1 == ids).all()
    mp = np.array([3, 100, 192], dtype=np.uint32)
    want = oracle.libvdbscan(x, y, [EPS] * 3, mp)
    for budget in (0, 4 * max(int(off[-1]) // 3, 400)):  # one tile; several
        kw = {"table_budget_bytes": budget} if budget else {}
        got = vd.cluster(x, y, [EPS] * 3, mp, path=vd.PATH_TABLE, precision=prec, **kw)
        assert (got == want).all(), (name, budget)
