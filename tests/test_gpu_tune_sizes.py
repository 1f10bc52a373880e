"""Autotuner keys: sets whose point counts differ by a little are one workload
and are tuned once, whichever engine they go to."""
import numpy as np
import pytest

import variantdbscan_amd as vd
from variantdbscan_amd import _lib

pytestmark = pytest.mark.gpu

N = 141_000  # 131,072 points are where tuning begins; 2^17.125 = 142,937


def _points(n):
    r = np.random.Generator(np.random.PCG64(23))
    x, y = r.uniform(0.0, 120.0, N + 64), r.uniform(0.0, 120.0, N + 64)
    x[:2], y[:2] = [0.0, 120.0], [0.0, 120.0]  # the extent of every set
    return x[:n], y[:n]


CALLS = {
    "batch": lambda x, y: vd.cluster(x, y, [0.5, 0.7], [4, 9], path=vd.PATH_BATCH),
    "table": lambda x, y: vd.cluster(x, y, 0.5, 4, path=vd.PATH_TABLE),
    "fused, float32": lambda x, y: vd.cluster(x, y, 0.5, 4, path=vd.PATH_FUSED,
                                              precision=vd.PREC_FP32_RECHECK),
    "counts": lambda x, y: vd.neighbor_counts(x, y, 0.5),
    "reuse": lambda x, y: vd.cluster(x, y, [0.5, 0.5], [4, 9], reuse=True),
}


@pytest.mark.parametrize("call", CALLS)
def test_near_sizes_are_tuned_once(call):
    CALLS[call](*_points(N))
    print(call, "first size done", flush=True)
    tuned = _lib.tuning()["tuned_in_process"]
    for n in (N + 1, N + 17, N + 64, N - 500):
        CALLS[call](*_points(n))
        assert _lib.tuning()["tuned_in_process"] == tuned, n
