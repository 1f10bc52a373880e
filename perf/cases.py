"""Performance cases of the clustering library: what its users have it do.

A case is a dict: `entry` (which public entry point is called), `shape` (the
point cloud, as variantdbscan_amd/datasets.py describes them), `n` points (per
call; `sets` datasets share them in multi-dataset calls), and the entry's own
options. Every seed gives another point cloud of the same shape: blob centres,
widths and noise are all drawn from it, in float64 on the GPU, longitudes and
latitudes in degrees.

Entries:
  host      VariantDBSCAN(...): host arrays in, host labels out
  cluster   cluster_device(...): points and labels in device memory
  multi     cluster_multi_device(...): many datasets in one call
  table     vdb_neighbor_table on device pointers: the CSR table with its d2
  counts    vdb_neighbor_counts on device pointers
"""
import ctypes
import math

import numpy as np
import torch

import variantdbscan_amd as vd
from variantdbscan_amd import _lib

GRID64_EPS = "0.2,0.3,0.4,0.5,0.6,0.7,0.8,0.9"
GRID64_MINPTS = "4,6,8,12,16,24,32,48"
GRID16_EPS = "0.25,0.5,0.75,1.0"
GRID16_MINPTS = "4,8,16,32"
BOX_AREA = 180.0 * 360.0


def listed():
    """eps and minpts lists are crossed: every eps with every minpts."""
    return [
        # a few hundred to a thousand points from a script, as the reference's
        # own example does it (two variants of a small CSV): latency only
        {"name": "host_1k_2v", "entry": "host", "shape": "plain", "n": 1000,
         "eps": "0.5,1.0", "minpts": "10"},
        # the plain workload: 10,000 points, one variant, drop-in call
        {"name": "host_10k_1v", "entry": "host", "shape": "plain", "n": 10_000,
         "eps": "1.0", "minpts": "4"},
        # a parameter study of one mid-sized set with the drop-in call
        {"name": "host_50k_16v", "entry": "host", "shape": "plain", "n": 50_021,
         "eps": GRID16_EPS, "minpts": GRID16_MINPTS},
        # the headline: 2M points under 64 variants, all in device memory
        {"name": "batch64_2m", "entry": "cluster", "shape": "aniso", "n": 2_000_000,
         "eps": GRID64_EPS, "minpts": GRID64_MINPTS, "border": 0, "path": 0},
        # one variant of the same set
        {"name": "single_2m", "entry": "cluster", "shape": "aniso", "n": 2_000_000,
         "eps": "0.5", "minpts": "8", "border": 0, "path": 0},
        # one variant of a large skewed set with a dense clump
        {"name": "skew_8m", "entry": "cluster", "shape": "skew", "n": 8_000_000,
         "eps": "0.3", "minpts": "10", "border": 0, "path": 0},
        # textbook labels (noise -1) for a parameter study of half a million points
        {"name": "standard_500k_16v", "entry": "cluster", "shape": "aniso", "n": 500_009,
         "eps": GRID16_EPS, "minpts": GRID16_MINPTS, "border": 1, "path": 0},
        # dense-region search: minpts beyond what neighbour lists hold, so the
        # library runs variant by variant
        {"name": "minpts100_1m", "entry": "cluster", "shape": "aniso", "n": 1_000_000,
         "eps": "0.4,0.6", "minpts": "100", "border": 0, "path": 0},
        # the neighbour-table engine: count, scan, fill, clusters from it
        {"name": "table_engine_2m", "entry": "cluster", "shape": "aniso", "n": 2_000_000,
         "eps": "0.3", "minpts": "8", "border": 0, "path": 2},
        # many uneven datasets under the same variants (a survey's tiles, days
        # of a year): 256 sets of 1k to 500k points
        {"name": "multi_256", "entry": "multi", "shape": "plain", "sets": 256, "median": 40_000,
         "eps": GRID16_EPS, "minpts": GRID16_MINPTS},
        # the neighbour table itself with squared distances, for a caller's own
        # algorithm
        {"name": "table_100k_d2", "entry": "table", "shape": "plain", "n": 100_003, "eps": "0.5",
         "precision": 0},
        # neighbourhood sizes (density maps), float32 screening
        {"name": "counts_1m_f32", "entry": "counts", "shape": "aniso", "n": 1_000_000,
         "eps": "0.4", "precision": 1},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _some(rng, values, most):
    k = rng.randint(1, most)
    return sorted(rng.sample(values, k))


def draw(rng):
    entry = rng.choice(("host", "host", "cluster", "cluster", "standard", "minpts", "engine",
                        "multi", "table", "counts"))
    eps_all = [round(0.2 + 0.05 * i, 2) for i in range(17)]
    mp_all = [2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48, 64]

    def grid(k, j):
        return (",".join("%g" % e for e in _some(rng, eps_all, k)),
                ",".join("%d" % m for m in _some(rng, mp_all, j)))

    if entry == "host":
        e, m = grid(4, 4)
        return {"entry": "host", "shape": rng.choice(("plain", "aniso")),
                "n": _log(rng, 200, 200_000), "eps": e, "minpts": m}
    if entry == "cluster":
        e, m = grid(8, 8)
        return {"entry": "cluster", "shape": rng.choice(("plain", "aniso", "skew")),
                "n": _log(rng, 20_000, 4_000_000), "eps": e, "minpts": m, "border": 0, "path": 0}
    if entry == "standard":
        e, m = grid(4, 4)
        return {"entry": "cluster", "shape": rng.choice(("plain", "aniso")),
                "n": _log(rng, 5_000, 1_500_000), "eps": e, "minpts": m, "border": 1, "path": 0}
    if entry == "minpts":
        return {"entry": "cluster", "shape": rng.choice(("plain", "aniso")),
                "n": _log(rng, 50_000, 1_000_000), "eps": "%g" % rng.choice(eps_all[:9]),
                "minpts": "%d" % rng.randint(65, 400), "border": rng.randint(0, 1), "path": 0}
    if entry == "engine":
        return {"entry": "cluster", "shape": "aniso", "n": _log(rng, 100_000, 1_500_000),
                "eps": "%g" % round(rng.uniform(0.1, 0.3), 3), "minpts": "%d" % rng.randint(4, 40),
                "border": 0, "path": 2}
    if entry == "multi":
        return {"entry": "multi", "shape": "plain", "sets": rng.randint(2, 96),
                "median": _log(rng, 2_000, 50_000), "eps": GRID16_EPS, "minpts": GRID16_MINPTS}
    if entry == "table":
        return {"entry": "table", "shape": "plain", "n": _log(rng, 2_000, 120_000),
                "eps": "%g" % round(rng.uniform(0.2, 0.7), 3), "precision": rng.randint(0, 1)}
    return {"entry": "counts", "shape": rng.choice(("plain", "aniso")),
            "n": _log(rng, 20_000, 1_500_000), "eps": "%g" % round(rng.uniform(0.1, 0.6), 3),
            "precision": rng.randint(0, 1)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rand(g, n, lo, hi):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _mixture(g, comp, cx, cy, sx, sy, th):
    """One point per entry of comp: from Gaussian blob comp (redrawn until it
    lies in the box), uniform where comp is negative. Points are independent
    draws, so their order carries no structure."""
    n = comp.numel()
    x, y = _rand(g, n, -90.0, 90.0), _rand(g, n, -180.0, 180.0)
    todo = (comp >= 0).nonzero().reshape(-1)
    while todo.numel():
        k = comp[todo]
        u = torch.randn(todo.numel(), generator=g, device="cuda", dtype=torch.float64) * sx[k]
        v = torch.randn(todo.numel(), generator=g, device="cuda", dtype=torch.float64) * sy[k]
        c, s = torch.cos(th[k]), torch.sin(th[k])
        bx, by = cx[k] + c * u - s * v, cy[k] + s * u + c * v
        x[todo], y[todo] = bx, by
        todo = todo[(bx.abs() > 90.0) | (by.abs() > 180.0)]
    return x.contiguous(), y.contiguous()


def _pick(g, n, weights):
    """n draws of an index by weight; the last weight stands for index -1."""
    edge = torch.cumsum(torch.tensor(weights, dtype=torch.float64, device="cuda"), 0)
    k = torch.searchsorted(edge, _rand(g, n, 0.0, float(edge[-1])), right=True)
    k = k.clamp_(max=len(weights) - 1)
    return torch.where(k == len(weights) - 1, torch.full_like(k, -1), k)


def _points(shape, n, seed):
    g = _gen(seed)
    if shape == "plain":  # 70% from 20 blobs of width 0.5, 30% uniform
        b = 20
        comp = _pick(g, n, [0.7 / b] * b + [0.3])
        sx = sy = torch.full((b,), 0.5, dtype=torch.float64, device="cuda")
        th = torch.zeros(b, dtype=torch.float64, device="cuda")
    elif shape == "aniso":  # 60% from 200 stretched blobs, Zipf weights, 40% uniform
        b = 200
        z = [(i + 1.0) ** -1.1 for i in range(b)]
        comp = _pick(g, n, [0.6 * w / sum(z) for w in z] + [0.4])
        sx, sy = (0.3 * torch.exp(0.5 * torch.randn(b, generator=g, device="cuda",
                                                    dtype=torch.float64)) for _ in range(2))
        th = _rand(g, b, 0.0, math.pi)
    else:  # skew: half uniform, 45% from 500 blobs of width 0.2, 5% in one 1 x 1 clump
        b = 500
        comp = _pick(g, n, [0.45 / b] * b + [0.55])
        sx = sy = torch.full((b,), 0.2, dtype=torch.float64, device="cuda")
        th = torch.zeros(b, dtype=torch.float64, device="cuda")
    x, y = _mixture(g, comp, _rand(g, b, -90.0, 90.0), _rand(g, b, -180.0, 180.0), sx, sy, th)
    if shape == "skew":
        k = (_rand(g, n, 0.0, 1.0) < 0.05 / 0.55) & (comp < 0)
        c = _rand(g, 2, 0.0, 1.0).tolist()
        x = torch.where(k, _rand(g, n, 0.0, 1.0) + (c[0] * 178.0 - 90.0), x)
        y = torch.where(k, _rand(g, n, 0.0, 1.0) + (c[1] * 358.0 - 180.0), y)
    return x, y


def _multi_sizes(case):
    """Dataset sizes: lognormal about the median, 1k to 500k. The same for
    every seed, so that a case is always the same amount of work."""
    r = np.random.Generator(np.random.PCG64(5))
    s = np.exp(math.log(case["median"]) + r.normal(0.0, 1.15, case["sets"]))
    return np.clip(np.round(s), 1_000, 500_000).astype(np.int64)


def _multi_points(case, seed):
    """Datasets of the plain shape, 5 to 100 blobs each."""
    g = _gen(seed)
    sizes = torch.from_numpy(_multi_sizes(case)).cuda()
    sets = case["sets"]
    nb = torch.randint(5, 101, (sets,), generator=g, device="cuda")
    ds = torch.repeat_interleave(torch.arange(sets, device="cuda"), sizes)
    n = ds.numel()
    k = (_rand(g, n, 0.0, 1.0) * nb[ds]).long()
    comp = torch.where(_rand(g, n, 0.0, 1.0) < 0.7, ds * 100 + k, torch.full_like(k, -1))
    b = sets * 100
    w = torch.full((b,), 0.5, dtype=torch.float64, device="cuda")
    return _mixture(g, comp, _rand(g, b, -90.0, 90.0), _rand(g, b, -180.0, 180.0), w, w,
                    torch.zeros_like(w))


def _variants(case):
    eps = [float(t) for t in case["eps"].split(",")]
    mp = [int(t) for t in case["minpts"].split(",")]
    e = np.array([a for a in eps for _ in mp], dtype=np.float64)
    m = np.array([b for _ in eps for b in mp], dtype=np.uint32)
    return e, m


def prepare(case, seed):
    entry = case["entry"]
    if entry == "multi":
        x, y = _multi_points(case, seed)
        offsets = np.concatenate([[0], np.cumsum(_multi_sizes(case))]).astype(np.uint64)
        eps, mp = _variants(case)
        labels = torch.empty(x.numel() * len(eps), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return {"case": case, "x": x, "y": y, "offsets": offsets, "eps": eps, "minpts": mp,
                "labels": labels}
    x, y = _points(case["shape"], case["n"], seed)
    state = {"case": case, "x": x, "y": y}
    n = case["n"]
    if entry == "host":
        state["eps"], state["minpts"] = _variants(case)
        state["x"], state["y"] = x.cpu().numpy(), y.cpu().numpy()
    elif entry == "cluster":
        state["eps"], state["minpts"] = _variants(case)
        state["labels"] = torch.empty((len(state["eps"]), n), dtype=torch.int32, device="cuda")
    elif entry == "counts":
        state["counts"] = torch.empty(n, dtype=torch.int32, device="cuda")
    else:  # table: buffers of a fixed capacity, kept from call to call
        state["offsets"] = torch.empty(n + 1, dtype=torch.int64, device="cuda")
        state["ids"] = torch.zeros(_capacity(case), dtype=torch.int32, device="cuda")
        state["d2"] = torch.zeros(_capacity(case), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()  # the library works on a stream of its own
    return state


# -------------------------------------------------------------------- passes
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _check(rc):
    if rc:
        raise RuntimeError("vdbscan error %d" % rc)


def run(state):
    case = state["case"]
    entry = case["entry"]
    if entry == "host":
        return vd.VariantDBSCAN(state["eps"], state["minpts"], state["x"], state["y"])
    if entry == "cluster":
        vd.cluster_device(state["x"].data_ptr(), state["y"].data_ptr(), case["n"], state["eps"],
                          state["minpts"], state["labels"].data_ptr(), path=case["path"],
                          stats=False, border=case["border"])
        return state["labels"]
    if entry == "multi":
        vd.cluster_multi_device(state["x"].data_ptr(), state["y"].data_ptr(), state["offsets"],
                                state["eps"], state["minpts"], state["labels"].data_ptr())
        return state["labels"]
    if entry == "counts":
        _check(_lib.load().vdb_neighbor_counts(
            _ptr(state["x"]), _ptr(state["y"]), case["n"], float(case["eps"]),
            _ptr(state["counts"]), _lib.DEVICE_PTRS, case["precision"], None))
        return state["counts"]
    total = ctypes.c_uint64(0)
    _check(_lib.load().vdb_neighbor_table(
        _ptr(state["x"]), _ptr(state["y"]), case["n"], float(case["eps"]), _ptr(state["offsets"]),
        _ptr(state["ids"]), _ptr(state["d2"]), state["ids"].numel(), ctypes.byref(total),
        _lib.DEVICE_PTRS, case["precision"], None))
    if total.value > state["ids"].numel():
        raise RuntimeError("the table needs %d entries" % total.value)
    return {"offsets": state["offsets"], "ids": state["ids"], "d2": state["d2"]}


def _expected_pairs(n, eps):
    """Neighbour pairs of the plain shape (self pairs included), on average:
    inside a blob two points are within eps with probability 1 - exp(-(eps/2s)^2)."""
    blob = 0.7 * n / 20
    inside = 20 * blob * blob * (1.0 - math.exp(-(eps / (2 * 0.5)) ** 2))
    cover = math.pi * eps * eps / BOX_AREA
    return n + inside + (n * n - 20 * blob * blob) * cover


def _capacity(case):
    """Table entries a caller allows for: overlapping blobs add some pairs to
    the average (the entries past the table stay zero)."""
    return int(1.5 * _expected_pairs(case["n"], float(case["eps"]))) + 1024


def work(case):
    """Each input read once, each output written once."""
    entry = case["entry"]
    if entry == "table":
        n = case["n"]
        return {"bytes": 16.0 * n + 8.0 * (n + 1) + 8.0 * _expected_pairs(n, float(case["eps"])),
                "flops": 0.0}
    if entry == "counts":
        return {"bytes": 20.0 * case["n"], "flops": 0.0}
    n = int(_multi_sizes(case).sum()) if entry == "multi" else case["n"]
    return {"bytes": 16.0 * n + 4.0 * n * len(_variants(case)[0]), "flops": 0.0}


# --------------------------------------------------------------- exact values
def exact(case, seed):
    """The table's squared distances in binary64, in the table's own order:
    rows by caller index, inside a row the points by grid cell (half an eps
    wide, column-major), inside a cell by the reference's visit order."""
    if case["entry"] != "table":
        return None
    n, eps = case["n"], float(case["eps"])
    x, y = _points(case["shape"], n, seed)
    bins = []
    for v in (x, y):
        lo, hi = float(v.min()), max(float(v.max()), 2.2250738585072014e-308)
        width = (hi - lo) * 1.01
        bins.append(torch.floor((v + (-lo if lo > 0 else abs(lo))) / width * 300.0).long())
    rank = torch.sort(bins[0] * 300 + bins[1], stable=True)[1]
    w = eps * (1.0 + 2.0 ** -24) / 2
    cx = torch.floor((x[rank] - x.min()) / w).long()
    cy = torch.floor((y[rank] - y.min()) / w).long()
    order = rank[torch.sort(cx * (int(cy.max()) + 2) + cy, stable=True)[1]]
    xs, ys = x[order], y[order]
    out, rows = [], max(1, (1 << 26) // n)
    for a in range(0, n, rows):
        dx = x[a:a + rows, None] - xs[None, :]
        dy = y[a:a + rows, None] - ys[None, :]
        s = dx * dx + dy * dy
        out.append(s[torch.sqrt(s) <= eps])
    d2 = torch.zeros(_capacity(case), dtype=torch.float64, device="cuda")
    found = torch.cat(out)
    d2[:found.numel()] = found
    return {"offsets": None, "ids": None, "d2": d2}
