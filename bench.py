#!/usr/bin/env python3
"""Benchmark of the VariantDBSCAN hot path on one MI355X.

Headline (`value`): variant-clusterings per second, with exact labels, of the
batched engine on 2,000,000 points x 64 variants (eps 0.2..0.9 step 0.1 x
minpts {4,6,8,12,16,24,32,48}); points and labels resident in HBM; one step =
one call clustering all 64 variants.

Also measured in the same run (each in its own timed region, none of them
`value`):
  * `batch_standard_border`: the same batched call under the standard border
    rule (textbook DBSCAN labels, noise -1).
  * `end_to_end_host`: the drop-in libVDBSCAN call on the same 2M x 64
    workload from host arrays (upload and the 512 MB label copy included).
  * `roofline`: the CSR neighbour-table fill kernel at eps 0.5 on the same
    points (ids only, FP64), algorithmic bytes per launch over its HIP-event
    duration against 8 TB/s; `table_build` adds the count and scan kernels.
  * `plain_fp64`: the per-variant FP64 engines, one variant per eps level
    (minpts 8): the fused engine (no table, the library's per-variant
    default) and the CSR table engine; `ratio_vs_plain` = value / fused
    variants/s, `ratio_vs_plain_table` = value / table variants/s.
  * `skew_8m`: 8,000,000 points with a dense 1x1 deg clump, eps 0.3, minpts
    10, table engine in FP64 and in FP32 with the binary64 recheck (rechecked
    pair count and fraction).
  * `multi_256`: 256 uneven datasets (17.8M points) x 16 variants in one
    vdb_cluster_multi call, datasets x variants per second.
  * `cpu_baseline`: the reference library (compiled from its sources into
    oracle/_ref) on a 100,000-point random subsample of the 2M points, all 64
    variants in one call, on the host's cores.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu]
       [--no-table] [--no-plain] [--no-extra] [--no-standard] [--only batch|table]
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "variant-clusterings/sec at exact labels, 2M pts×64 variants; neighbor-table HBM GB/s"
HBM_PEAK_GBS = 8000.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def table_bytes(n, pairs, k_cuts=1, with_dist=False):
    """Algorithmic bytes of one CSR neighbour-table build:
    16N read points + 4N*K counts + 16N scan (counts in, int64 offsets out)
    + 24N fill (points + offsets re-read) + P*(4 [+4]) ids (and distances)."""
    return 16 * n + 4 * n * k_cuts + 16 * n + 24 * n + pairs * (4 + (4 if with_dist else 0))


def fill_bytes(n, pairs):
    """Algorithmic bytes of the fill kernel alone: 24N in + 4P ids out."""
    return 24 * n + 4 * pairs


# batched-engine kernels timed for the headline roofline
BATCH_KERNELS = ("k_knn", "k_sweep", "k_test", "k_labels_all", "k_rows_all", "k_labels_j",
                 "k_rows_from_pos", "k_roots_min", "k_pair_elig", "k_pair_scatter", "k_pairs",
                 "k_pair_count")


def batch_kernel_bytes(name, info, W):
    """Algorithmic bytes per step of a batched-engine kernel (summed over its
    launches; None for k_knn, k_test and k_roots_min, whose traffic follows
    the data). info: vdb_batch_info; W: fine-grid window width (2R+1), an
    upper bound of the window's rows (strips of columns).
      k_sweep       per record read (a pair entering at its level, for up to 8
                    minpts values, or carried from an earlier one) 12; per
                    record the two cells' parents (8 per minpts value); per
                    record written (carried on or a test slot) 12
      k_labels_all  per point: rank, cell, packed core levels (12), per
                    variant its cell label in and staged label out (8 V);
                    the list walk of non-core points is not counted
      k_rows_all    per point: its position (4), dataset bounds (8), its V
                    staged labels in and V output labels out (8 V)
      k_labels_j    per point: rank, cell, list index (12), its core level (1),
                    the 8 slots' cell labels (32) and its 8 staged labels (32)
      k_rows_from_pos per point: its position (4), dataset bounds (8), its
                    8 staged labels (32) and 8 output labels (32)
      k_pair_elig   per cell pair: its record (12), both cells' core levels
                    for each minpts value (2 J), a level byte per minpts value
                    out (8 per plane of 8 values)
      k_pair_scatter per cell pair: its record (12) and its level bytes (8 per
                    plane); per record written (a pair entering at its
                    level) 12
      k_pairs       per cell: its window rows (8 W) and box (32); per stored
                    pair 12 bytes
      k_pair_count  per cell: window rows (8 W), box (32), count (4)"""
    n, J = info["points"], info["minpts_values"]
    nc, npairs = info["cells"], info["cell_pairs"]
    planes = -(-J // 8)
    V = info.get("snapshots") or info["levels"] * J  # one per requested (level, minpts)
    fr, ca, te = info.get("fresh_pairs", 0), info.get("carried_pairs", 0), info.get("test_records", 0)
    return {
        "k_sweep": ((12 + 8 * min(J, 8)) * (fr + ca) + 12 * (ca + te)) if fr + ca else None,
        "k_labels_all": (12 + 8 * V) * n,
        "k_rows_all": (12 + 8 * V) * n,
        "k_labels_j": 77 * n * -(-V // 8),
        "k_rows_from_pos": 76 * n * -(-V // 8),
        "k_pair_elig": npairs * (12 + 2 * J + 8 * planes),
        "k_pair_scatter": (npairs * (12 + 8 * planes) + 12 * fr) if fr else None,
        "k_pairs": nc * (8 * W + 32) + npairs * 12,
        "k_pair_count": nc * (8 * W + 36),
    }.get(name)


def check_digests(labels, eps, mp):
    """'64/64' when every variant's labels (device tensor, V x n) hash to the
    committed digest of tests/golden/full_size_digests.json (aniso_2m:
    the oracle's labels, matched to the compiled reference on the first
    500,000 points), else 'k/64'; None without the file."""
    import hashlib
    path = os.path.join(ROOT, "tests", "golden", "full_size_digests.json")
    if not os.path.exists(path):
        return None
    w = json.load(open(path))["workloads"]["aniso_2m"]["variants"]
    host = labels.cpu().numpy().astype("<u4")
    ok = 0
    for v in range(len(eps)):
        want = w["eps%.2f/mp%d" % (eps[v], mp[v])]["sha256"]
        ok += hashlib.sha256(host[v].tobytes()).hexdigest() == want
    return "%d/%d" % (ok, len(eps))


def host_cpu():
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        usable = len(os.sched_getaffinity(0))
    except AttributeError:
        usable = os.cpu_count()
    return model, os.cpu_count(), usable


def cpu_leg(x, y, eps, mp, dev, stream):
    """The reference library (compiled from its sources into oracle/_ref) on
    the host, per BASELINE's plan, on bounded samples of each workload (about
    half a minute in all). Every sample's time is scaled to the full workload
    by the ratio of exact pair counts (the reference's work is one candidate
    test per pair per query), counted by the library on the GPU. A
    single-variant reference call runs on one core (it parallelises across
    variants only, src/main.cpp:215-216)."""
    import torch
    from concurrent.futures import ThreadPoolExecutor
    import variantdbscan_amd as vd
    from variantdbscan_amd import datasets
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle
    threads = 16 if oracle.ref_available(16) else 8 if oracle.ref_available(8) else 1
    if not oracle.ref_available(1) or not oracle.ref_available(threads):
        return None
    model, nproc, usable = host_cpu()

    def pairs(px, py, e):
        return int(vd.neighbor_counts(px, py, e).sum(dtype=np.uint64))

    n = len(x)
    ns = 200_000
    xs, ys = x[:ns], y[:ns]
    sx, sy = datasets.skew_8m()
    s1x, s1y = sx[:1_000_000], sy[:1_000_000]
    px, py = datasets.plain_10k(seed=1)
    # pair counts of full workloads and samples (GPU)
    E = sorted(set(eps.tolist()))
    p_full = {e: pairs(x, y, e) for e in E}
    p_samp = {e: pairs(xs, ys, e) for e in E}
    p4_full, p4_samp = pairs(sx, sy, 0.3), pairs(s1x, s1y, 0.3)
    sets = datasets.multi_256()
    # the 16 datasets around the median size (the largest, up to 500k points,
    # would hold tens of GB of reference expansion stacks across 16 threads)
    order = np.argsort([len(s[0]) for s in sets], kind="stable")
    pick = sorted(order[len(sets) // 2 - 8: len(sets) // 2 + 8].tolist())
    E5, M5 = datasets.MULTI_EPS, datasets.MULTI_MINPTS
    eps5 = np.array([e for e in E5 for m in M5])
    mp5 = np.array([m for e in E5 for m in M5], dtype=np.uint32)
    p5 = [sum(pairs(s[0], s[1], e) for e in E5) for s in sets]
    del sx, sy
    log("cpu: reference (%s, %d usable cores): configs 1, 2, 4 in parallel, single-threaded" %
        (model, usable))
    jobs = {
        "config1": (px, py, [1.0], [4], 1),
        "config2": (xs, ys, [0.5], [8], 1),
        "config4": (s1x, s1y, [0.3], [10], 1),
    }
    with ThreadPoolExecutor(len(jobs)) as ex:
        fut = {k: ex.submit(oracle.run_reference, *v[:4], threads=v[4], timeout=600)
               for k, v in jobs.items()}
        sec = {k: f.result()[1] for k, f in fut.items()}
    log("cpu: reference config 3 sample, %d threads" % threads)
    _, sec3 = oracle.run_reference(xs, ys, eps, mp, threads=threads, timeout=600)
    log("cpu: reference config 5 sample (%d datasets), %d threads" % (len(pick), threads))
    sec5 = sum(oracle.run_reference(sets[d][0], sets[d][1], eps5, mp5, threads=threads,
                                    timeout=600)[1] for d in pick)
    V = len(eps)
    r3 = sum(p_full[e] for e in eps) / sum(p_samp[e] for e in eps)
    r2 = p_full[0.5] / p_samp[0.5]
    r4 = p4_full / p4_samp
    r5 = sum(p5) / sum(p5[d] for d in pick)
    # the GPU batched engine on the config-3 sample, for a like-for-like line
    gx = torch.from_numpy(xs).to(dev)
    gy = torch.from_numpy(ys).to(dev)
    gl = torch.empty(V * ns, dtype=torch.int32, device=dev)
    for _ in range(3):
        vd.cluster_device(gx.data_ptr(), gy.data_ptr(), ns, eps, mp, gl.data_ptr(),
                          path=vd.PATH_BATCH)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(3):
        vd.cluster_device(gx.data_ptr(), gy.data_ptr(), ns, eps, mp, gl.data_ptr(),
                          path=vd.PATH_BATCH)
    e1.record(stream)
    torch.cuda.synchronize()
    gms = e0.elapsed_time(e1) / 3
    return {
        "value": V / (sec3 * r3), "unit": "variant-clusterings/s", "cores": threads,
        "kind": "reference",
        "sample": "config 3 (2M points x 64 variants) timed on its first 200,000 points, all 64 "
                  "variants in one libVDBSCAN call (NSEARCHTHREADS=%d, parallel across "
                  "variants, greedy cluster reuse), %.2f s; scaled to 2M points by the pair-count "
                  "ratio %.1f (sum over the 64 variants' eps)" % (threads, sec3, r3),
        "cpu_model": model, "nproc": nproc, "usable_cores": usable,
        "sample_variants_per_s": V / sec3, "gpu_same_sample_variants_per_s": V / (gms / 1e3),
        "configs": {
            "config1": {"workload": "10,000 points, eps 1.0, minpts 4, one call (full size)",
                        "seconds": sec["config1"], "cores": 1},
            "config2": {"workload": "2M points, eps 0.5, minpts 8, one single-variant call",
                        "sample": "first 200,000 points", "sample_seconds": sec["config2"],
                        "pair_ratio": r2, "seconds_full_estimate": sec["config2"] * r2,
                        "variants_per_s": 1.0 / (sec["config2"] * r2), "cores": 1},
            "config4": {"workload": "8M points (skewed), eps 0.3, minpts 10, one call",
                        "sample": "first 1,000,000 points", "sample_seconds": sec["config4"],
                        "pair_ratio": r4, "seconds_full_estimate": sec["config4"] * r4,
                        "cores": 1},
            "config5": {"workload": "256 datasets x 16 variants, one call per dataset",
                        "sample": "the 16 datasets around the median size (%d to %d "
                                  "points)" % (min(len(sets[d][0]) for d in pick),
                                               max(len(sets[d][0]) for d in pick)),
                        "sample_seconds": sec5, "pair_ratio": r5,
                        "seconds_full_estimate": sec5 * r5,
                        "datasets_x_variants_per_s": len(sets) * len(eps5) / (sec5 * r5),
                        "cores": threads},
        },
    }


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-table", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--no-extra", action="store_true",
                    help="skip the skew_8m and multi_256 side measurements")
    ap.add_argument("--only", choices=["batch", "table"], default=None)
    ap.add_argument("--no-standard", action="store_true",
                    help="skip the standard-border-rule timing of the batch leg")
    ap.add_argument("--table-steps", type=int, default=4,
                    help="table-path calls; the first (allocation, autotuning) is untimed")
    ap.add_argument("--kernel-steps", type=int, default=3,
                    help="steps per kernel of the headline roofline's per-kernel timing")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run a 1 GiB device copy first in the batch and table legs (HBM "
                         "counter calibration)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path "
              "(--gpus %d requested)" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import torch
    import variantdbscan_amd as vd
    from variantdbscan_amd import datasets

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    L = vd._lib.load()
    # a stream of its own (default priority): the library replays its launch
    # sequences from HIP graphs, and the NULL stream cannot be captured
    stream = torch.cuda.Stream(device=dev)
    torch.cuda.set_stream(stream)
    L.vdb_set_stream(stream.cuda_stream)

    x, y = datasets.aniso_2m()
    n = len(x)
    E, M = datasets.BATCH64_EPS, datasets.BATCH64_MINPTS
    eps = np.array([e for e in E for m in M])
    mp = np.array([m for e in E for m in M], dtype=np.uint32)
    V = len(eps)
    dx = torch.from_numpy(x).to(dev)
    dy = torch.from_numpy(y).to(dev)
    out = {}

    # ------------------------------------------------------------ batch
    if args.only in (None, "batch"):
        if args.calibrate_copy:
            # plain copy of known size (1 GiB read + 1 GiB written): the scale
            # of the HBM counters of the batched kernels' profile
            ca = torch.ones(1 << 28, dtype=torch.float32, device=dev)
            cb = torch.empty_like(ca)
            cb.copy_(ca)
            torch.cuda.synchronize()
            del ca, cb
        labels = torch.empty(V * n, dtype=torch.int32, device=dev)
        log("batch: warmup %d" % args.warmup)
        for _ in range(args.warmup):
            vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                              path=vd.PATH_BATCH)
        torch.cuda.synchronize()
        log("batch: timing %d steps" % args.steps)
        ev0 = torch.cuda.Event(enable_timing=True)
        ev1 = torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        ev0.record(stream)
        # the drop-in call as a caller makes it: no phase statistics (their
        # event reads add host waits)
        for _ in range(args.steps):
            vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                              path=vd.PATH_BATCH, stats=False)
        ev1.record(stream)
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        ms_step = ev0.elapsed_time(ev1) / args.steps
        value = V / (ms_step / 1e3)
        # phase times and the engine used, from calls made after the timed ones
        phases = [vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                                    path=vd.PATH_BATCH) for _ in range(3)]
        assert all(p["path_used"] == vd.PATH_BATCH for p in phases)
        avg = {k: float(np.mean([p[k] for p in phases])) for k in
               ("ms_total", "ms_prepare", "ms_count", "ms_uf", "ms_labels")}
        out.update(value=value, ms_per_step=ms_step, wall_s=wall, batch_phases_ms=avg)
        log("batch: %.3f ms/step -> %.1f variants/s" % (ms_step, value))

        # Roofline of the headline step: every launch of each batched kernel
        # timed with HIP events on the library's stream over further steps
        # of the same call (graph replay is off while a kernel is timed);
        # the dominant kernel's algorithmic bytes per launch over its average
        # launch time.
        info = vd._lib.batch_info()
        d0 = min(E) / np.sqrt(2.0) * (1.0 - 2.0 ** -20)
        W = 2 * int(np.ceil(max(E) * (1.0 + 2.0 ** -30) / d0)) + 1
        per = {}
        for kname in BATCH_KERNELS:
            vd._lib.time_kernel(kname)
            for _ in range(args.kernel_steps):
                vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                                  path=vd.PATH_BATCH)
            ms, launches = vd._lib.kernel_time()
            vd._lib.time_kernel(None)
            if launches:
                lps = launches / args.kernel_steps
                bstep = batch_kernel_bytes(kname, info, W)
                per[kname] = {"ms_per_step": ms / args.kernel_steps,
                              "launches_per_step": lps,
                              "ms_per_launch": ms / launches,
                              # average over the step's launches
                              "algorithmic_bytes": None if bstep is None else bstep / lps}
        dom = max(per, key=lambda k: per[k]["ms_per_step"])
        out["batch_kernels"] = per
        out["batch_info"] = info
        rec = per[dom]
        if rec["algorithmic_bytes"] is not None:
            ach = rec["algorithmic_bytes"] / (rec["ms_per_launch"] / 1e3) / 1e9
            # HBM bytes per launch from the calibrated FETCH_SIZE/WRITE_SIZE
            # passes over this workload, recorded under profiles/
            traffic, tsrc = None, None
            tf = os.path.join(ROOT, "profiles", "hbm_counters_%s_aniso2m_batch64.json" % dom)
            if os.path.exists(tf):
                traffic = json.load(open(tf)).get("traffic_bytes")
                tsrc = os.path.relpath(tf, ROOT)
            out["roofline"] = {"bound": "hbm", "achieved": ach, "peak": HBM_PEAK_GBS,
                               "unit": "GB/s", "frac": ach / HBM_PEAK_GBS, "traffic": traffic,
                               "traffic_source": tsrc,
                               "kernel": dom, "algorithmic_bytes": rec["algorithmic_bytes"],
                               "ms_per_launch": rec["ms_per_launch"],
                               "ms_per_step": rec["ms_per_step"],
                               "workload": "the headline step (2M points x 64 variants)"}
        log("batch: dominant kernel %s, %.3f ms per step (%.1f launches)" %
            (dom, rec["ms_per_step"], rec["launches_per_step"]))
        labels_ok = check_digests(labels.view(V, n), eps, mp)
        if labels_ok is not None:
            out["labels_match_reference"] = labels_ok

        # spot check against the per-variant engine on two variants
        chk = [0, V - 1]
        ref = torch.empty(len(chk) * n, dtype=torch.int32, device=dev)
        vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps[chk], mp[chk], ref.data_ptr(),
                          path=vd.PATH_FUSED)
        lab = labels.view(V, n)[chk]
        out["labels_match_per_variant_engine"] = bool(torch.equal(lab, ref.view(len(chk), n)))

        # the same call under the standard border rule (textbook DBSCAN
        # labels), with the same spot check
        for _ in range(0 if args.no_standard else args.warmup):
            vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                              path=vd.PATH_BATCH, border=vd.BORDER_STANDARD)
        if not args.no_standard:
            sa = torch.cuda.Event(enable_timing=True)
            sb = torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            sa.record(stream)
            for _ in range(args.steps):
                vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps, mp, labels.data_ptr(),
                                  path=vd.PATH_BATCH, border=vd.BORDER_STANDARD, stats=False)
            sb.record(stream)
            torch.cuda.synchronize()
            ms_std = sa.elapsed_time(sb) / args.steps
            vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, eps[chk], mp[chk], ref.data_ptr(),
                              path=vd.PATH_FUSED, border=vd.BORDER_STANDARD)
            lab = labels.view(V, n)[chk]
            out["batch_standard_border"] = {
                "ms_per_step": ms_std, "variants_per_s": V / (ms_std / 1e3),
                "labels_match_per_variant_engine": bool(torch.equal(lab, ref.view(len(chk), n)))}
            log("batch, standard border rule: %.3f ms/step" % ms_std)
        del labels, ref
        L.vdb_release()
        torch.cuda.empty_cache()

    # --------------------------------------------- neighbour-table roofline
    if args.only in (None, "table") and not args.no_table:
        # the table leg reads the device time of each kernel phase from HIP
        # events the library records on this stream
        if args.calibrate_copy:
            # plain copy of known size: 1 GiB read + 1 GiB written
            ca = torch.ones(1 << 28, dtype=torch.float32, device=dev)
            cb = torch.empty_like(ca)
            cb.copy_(ca)
            torch.cuda.synchronize()
            del ca, cb
        lab1 = torch.empty(n, dtype=torch.int32, device=dev)
        tphases = []
        for i in range(args.table_steps):
            st = vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, [0.5], [8], lab1.data_ptr(),
                                   path=vd.PATH_TABLE)
            tphases.append(st)
            log("table: step %d count %.2f scan %.2f fill %.2f ms, %d pairs, %d tile(s)" %
                (i, st["ms_count"], st["ms_scan"], st["ms_fill"], st["pairs"], st["tiles"]))
        torch.cuda.synchronize()
        t = tphases[-1] if len(tphases) == 1 else tphases[1]
        P = int(t["pairs"])
        fill_ms = float(np.mean([p["ms_fill"] for p in tphases[1:] or tphases]))
        cnt_ms = float(np.mean([p["ms_count"] for p in tphases[1:] or tphases]))
        scan_ms = float(np.mean([p["ms_scan"] for p in tphases[1:] or tphases]))
        fb = fill_bytes(n, P)
        achieved = fb / (fill_ms / 1e3) / 1e9
        tb = table_bytes(n, P)
        tab_gbs = tb / ((cnt_ms + scan_ms + fill_ms) / 1e3) / 1e9
        # HBM bytes per launch from the calibrated FETCH_SIZE/WRITE_SIZE passes
        # recorded under profiles/ for this kernel and workload
        traffic = None
        tf = os.path.join(ROOT, "profiles", "hbm_counters_k_fill.json")
        if os.path.exists(tf):
            traffic = json.load(open(tf)).get("traffic_bytes")
        out["roofline_table_fill"] = {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                           "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
                           "traffic_source": "profiles/hbm_counters_k_fill.md",
                           "kernel": "k_fill<0, false, false> (CSR neighbour-table fill, FP64, "
                                     "rows staged in LDS)",
                           "workload": "2M points, eps 0.5, %d pairs, %d tile(s)" %
                           (P, t["tiles"]),
                           "algorithmic_bytes": fb, "ms_per_launch": fill_ms}
        out["table_build"] = {"count_ms": cnt_ms, "scan_ms": scan_ms, "fill_ms": fill_ms,
                              "pairs": P, "algorithmic_bytes": tb, "achieved_gbs": tab_gbs,
                              "frac": tab_gbs / HBM_PEAK_GBS}
        del lab1
        L.vdb_release()
        torch.cuda.empty_cache()

    # ------------------------------------------------ plain per-variant path
    if args.only is None and not args.no_plain:
        # one variant per eps level (minpts 8, the cost is set by eps), each
        # clustered on its own by the per-variant FP64 engines: fused (no
        # table; the library's per-variant default) and CSR table
        lab1 = torch.empty(n, dtype=torch.int32, device=dev)
        res = {}
        for path, nm in ((vd.PATH_FUSED, "fused"), (vd.PATH_TABLE, "table")):
            per = {}
            # largest eps first: its table sizes the pooled buffer the others reuse
            for e in sorted(E, reverse=True):
                # first call of a workload runs the grid autotuner: untimed
                vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, [e], [8], lab1.data_ptr(),
                                  path=path)
                torch.cuda.synchronize()
                ea = torch.cuda.Event(enable_timing=True)
                eb = torch.cuda.Event(enable_timing=True)
                ea.record(stream)
                vd.cluster_device(dx.data_ptr(), dy.data_ptr(), n, [e], [8], lab1.data_ptr(),
                                  path=path)
                eb.record(stream)
                torch.cuda.synchronize()
                per[e] = ea.elapsed_time(eb)
                log("plain fp64 %s path eps %.1f: %.1f ms" % (nm, e, per[e]))
            ms = [per[e] for e in E]
            res[nm] = {"variants_per_s": len(E) / (sum(ms) / 1e3), "ms_per_eps_level": ms}
            L.vdb_release()
            torch.cuda.empty_cache()
        out["plain_fp64"] = {"variants_per_s": res["fused"]["variants_per_s"],
                             "engine": "fused per-variant (grid, core test, components over "
                                       "cells, borders, labels)",
                             "ms_per_eps_level": res["fused"]["ms_per_eps_level"],
                             "table_engine": res["table"],
                             "sample": "minpts 8 at each of the 8 eps levels"}
        if "value" in out:
            out["ratio_vs_plain"] = out["value"] / res["fused"]["variants_per_s"]
            out["ratio_vs_plain_table"] = out["value"] / res["table"]["variants_per_s"]
        del lab1

    # ------------------------------------------ other workloads (not `value`)
    if args.only is None and not args.no_extra:
        del dx, dy
        L.vdb_release()
        torch.cuda.empty_cache()
        # the drop-in call end to end: host arrays in, labels out through
        # libVDBSCAN (upload, batched engine, label copy to pageable memory)
        ret = np.empty(V * n, dtype=np.uint32)
        hx, hy = np.ascontiguousarray(x), np.ascontiguousarray(y)
        he = np.ascontiguousarray(eps, dtype=np.float64)
        hm = np.ascontiguousarray(mp, dtype=np.uint32)

        def drop_in():
            rc = L.libVDBSCAN(hx.ctypes.data, hy.ctypes.data, n, he.ctypes.data,
                              hm.ctypes.data, V, 70, ret.ctypes.data, False)
            assert rc == 0, vd._lib.last_error()

        drop_in()
        reps = 3
        t0 = time.perf_counter()
        for _ in range(reps):
            drop_in()
        e2e = (time.perf_counter() - t0) / reps
        out["end_to_end_host"] = {"entry": "libVDBSCAN (host arrays, pageable)",
                                  "s_per_call": e2e, "variants_per_s": V / e2e}
        log("libVDBSCAN end to end: %.1f ms per call -> %.0f variants/s" % (e2e * 1e3, V / e2e))
        del ret
        L.vdb_release()
        # 8M points with a dense clump, eps 0.3, minpts 10: FP32 screening
        # with binary64 recheck against plain FP64
        sx, sy = datasets.skew_8m()
        dsx = torch.from_numpy(sx).to(dev)
        dsy = torch.from_numpy(sy).to(dev)
        lab = torch.empty(len(sx), dtype=torch.int32, device=dev)
        rec = {}
        for prec, nm in ((vd.PREC_FP64, "fp64"), (vd.PREC_FP32_RECHECK, "fp32_recheck")):
            for rep in range(2):
                st = vd.cluster_device(dsx.data_ptr(), dsy.data_ptr(), len(sx), [0.3], [10],
                                       lab.data_ptr(), path=vd.PATH_TABLE, precision=prec)
            rec[nm] = {"ms_total": st["ms_total"], "ms_count": st["ms_count"],
                       "ms_fill": st["ms_fill"], "pairs": st["pairs"],
                       "rechecked": st["rechecked"]}
            log("skew_8m table path %s: %.1f ms, rechecked %d" % (nm, st["ms_total"],
                                                                 st["rechecked"]))
        st = vd.cluster_device(dsx.data_ptr(), dsy.data_ptr(), len(sx), [0.3], [10],
                               lab.data_ptr(), path=vd.PATH_AUTO)
        rec["auto_ms_total"] = st["ms_total"]
        rec["recheck_fraction"] = rec["fp32_recheck"]["rechecked"] / max(1, rec["fp32_recheck"]["pairs"])
        out["skew_8m"] = rec
        del dsx, dsy, lab
        L.vdb_release()
        torch.cuda.empty_cache()
        # 256 uneven datasets x 16 variants in one call
        sets = datasets.multi_256()
        E5, M5 = datasets.MULTI_EPS, datasets.MULTI_MINPTS
        eps5 = np.array([e for e in E5 for m in M5])
        mp5 = np.array([m for e in E5 for m in M5], dtype=np.uint32)
        offs = np.zeros(len(sets) + 1, dtype=np.uint64)
        offs[1:] = np.cumsum([len(s[0]) for s in sets])
        mx = torch.from_numpy(np.concatenate([s[0] for s in sets])).to(dev)
        my = torch.from_numpy(np.concatenate([s[1] for s in sets])).to(dev)
        ml = torch.empty(int(offs[-1]) * len(eps5), dtype=torch.int32, device=dev)
        for rep in range(3):
            st = vd.cluster_multi_device(mx.data_ptr(), my.data_ptr(), offs, eps5, mp5,
                                         ml.data_ptr())
        out["multi_256"] = {"datasets": len(sets), "points": int(offs[-1]),
                            "variants": len(eps5), "ms_total": st["ms_total"],
                            "datasets_x_variants_per_s": len(sets) * len(eps5) /
                            (st["ms_total"] / 1e3)}
        log("multi_256: %.1f ms -> %.0f datasets x variants / s" %
            (st["ms_total"], out["multi_256"]["datasets_x_variants_per_s"]))
        del mx, my, ml
        L.vdb_release()
        torch.cuda.empty_cache()

    # ----------------------------------------------------------- CPU leg
    if args.only is None and not args.no_cpu:
        out["cpu_baseline"] = cpu_leg(x, y, eps, mp, dev, stream)

    line = {
        "metric": METRIC,
        "value": out.get("value"),
        "unit": "variant-clusterings/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": out.get("ms_per_step"),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded generator, variantdbscan_amd/datasets.py)",
        "config": {"workload": "aniso_2m: 2,000,000 points (60% from 200 anisotropic blobs, "
                               "40% uniform) x 64 variants (eps 0.2..0.9 x minpts 4..48), "
                               "batched engine, inputs and labels in HBM",
                   "n_points": n, "variants": V, "eps": E, "minpts": M},
        "roofline": out.get("roofline"),
        "cpu_baseline": out.get("cpu_baseline"),
    }
    for k in ("labels_match_reference", "batch_kernels", "batch_info", "roofline_table_fill",
              "ratio_vs_plain", "ratio_vs_plain_table", "plain_fp64", "table_build",
              "batch_standard_border", "end_to_end_host",
              "skew_8m", "multi_256", "batch_phases_ms",
              "labels_match_per_variant_engine", "wall_s"):
        if k in out:
            line[k] = out[k]
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
