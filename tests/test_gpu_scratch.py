"""Pooled device memory of small batched calls: the test lists follow the call's
cell pairs, not the largest grid of the level kernels."""
import ctypes

import numpy as np
import pytest

import oracle

import variantdbscan_amd as vd
from variantdbscan_amd import _lib

pytestmark = pytest.mark.gpu


def _free_bytes():
    H = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library links
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert H.hipDeviceSynchronize() == 0
    assert H.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


@pytest.mark.parametrize("n,nmp", [(1_000, 1), (1_000, 8), (50_000, 8)])
def test_small_calls_keep_little(n, nmp):
    r = np.random.Generator(np.random.PCG64(n))
    x, y = r.uniform(0, 10, n), r.uniform(0, 10, n)
    eps, mp = [0.5] * nmp, list(range(4, 4 + nmp))
    assert _lib.load().vdb_release() == 0
    before = _free_bytes()
    print(n, "points,", nmp, "minpts values", flush=True)
    got, st = vd.cluster(x, y, eps, mp, path=vd.PATH_BATCH, return_stats=True)
    assert st["path_used"] == vd.PATH_BATCH
    # about 400 bytes a point and as much a cell pair, in some 60 buffers
    assert before - _free_bytes() < 32 << 20
    if n == 1_000:
        assert (got == oracle.libvdbscan(x, y, eps, mp)).all()
