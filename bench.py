"""Benchmark: end-to-end octree build of 2^24 3D points on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload uniform|gauss]
    python bench.py --workload batch [--batch-count 4096]   (batched form)
    python bench.py --workload serve [--serve-rate 2000]    (served form)
    python bench.py --workload findleaf                     (point location)
    python bench.py --workload octree_text                  (text form of the octree)
    python bench.py --workload cellwalk                     (batched cell walks)
    python bench.py --workload gvd                          (GVD refinement, 2D polylines)

One step = the whole path (bounding box, FP32 quantize, 63-bit Morton keys,
radix sort, unique, Karras BRT with local splits, octree fill) over 2^24
float3 points that are already in HBM.  Prints one JSON line: sorted Morton
keys/s (whole job), the per-launch roofline of the dominant kernel (the
octree gather, or an onesweep sort pass where the LSD passes sorted), the
whole-path roofline against the path's algorithmic byte model, and the
serial CPU path (the oracle, one core) timed on a bounded sample.
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import os
import platform
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
METRIC = "sorted Morton keys/sec, end-to-end octree build at 2^24 pts; % HBM roofline"


def make_points(workload: str, n: int) -> tuple[np.ndarray, str]:
    """Synthetic inputs (seeded).  The conflict-cell workload returns labels
    through make_points.labels."""
    if workload == "conflict":
        from pgvd_amd.workloads import star_loops
        pts, labels = star_loops(n, loops=64, seed=4)
        make_points.labels = labels
        return pts, (f"3D conflict-cell build, {n} float3 on 64 star-shaped loops (256 vertices, "
                     f"radii 0.05-0.3, seed 4) with uint32 loop ids")
    if workload == "uniform":
        rng = np.random.default_rng(2)
        pts = rng.random((n, 3), dtype=np.float32) * 2 - 1
        return pts, f"3D octree build, {n} float3 uniform in [-1,1]^3 (seed 2)"
    if workload == "gauss":
        from pgvd_amd.workloads import gaussian_mixture
        return gaussian_mixture(n)
    raise SystemExit(f"unknown workload {workload}")


def algorithmic_bytes(n: int, m: int, O: int, dim: int, K: int, R: int, L: int = 0) -> dict:
    """Algorithmic HBM bytes of the path, term by term as a fixed byte model
    of its stages (whatever the kernels actually move): P = 4 dim point
    bytes, K key bytes, L label bytes, R = ceil(mbits/8) radix passes (the
    8-bit-digit convention, also when the bucket sort sorts in fewer passes
    over HBM), B = 16 + K compact BRT node bytes, N = 4 (2^dim + 1) octree
    node bytes.  The gather kernel performs the scan of local splits and the
    octree fill, so its figure is those two terms."""
    P = 4 * dim
    B = 16 + K
    N = 4 * ((1 << dim) + 1)
    parts = {
        "bbox": P * n,
        "encode": (P + K + L) * n,
        "sort": 2 * R * (K + L) * n,
        "unique": (K + L) * n + K * m,
        "brt": K * m + B * (m - 1),
        "splits": B * (m - 1) + 4 * m,
        "scan": 8 * m,
        "octree": (B + 8) * (m - 1) + N * O,
    }
    if L:
        parts["conflict"] = L * n + m // 8
    parts["total"] = sum(parts.values())
    parts["sort_pass"] = 2 * (K + L) * n
    parts["gather"] = parts["scan"] + parts["octree"]
    return parts


def cpu_baseline(pts: np.ndarray, bits: int, sample: int, labels=None) -> dict:
    import oracle
    L = oracle.lib()
    sub = np.ascontiguousarray(pts[:sample])
    try:
        os.sched_setaffinity(0, {sorted(os.sched_getaffinity(0))[0]})
        pinned = True
    except (AttributeError, OSError):
        pinned = False
    m = C.c_int64()
    t0 = time.perf_counter()
    if labels is None:
        osz = L.oracle_run_pipeline(sub.reshape(-1), sub.shape[0], sub.shape[1], bits, C.byref(m))
    else:     # quantize, then the serial path with the point-label conflict pass
        osz = oracle.build(oracle.quantize(sub, 1 << bits), bits,
                           labels=np.ascontiguousarray(labels[:sample]))["octree_size"]
    dt = time.perf_counter() - t0
    if osz < 0:
        raise RuntimeError("oracle pipeline failed")
    cpu = platform.processor() or platform.machine()
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    cpu = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {
        "value": sub.shape[0] / dt,
        "unit": "keys/s",
        "cores": 1,
        "kind": "port",
        "sample": (f"first {sub.shape[0]} points of the same workload, whole serial path "
                   f"(bbox, quantize, bit-serial Morton, comparison sort, unique, per-node BRT, "
                   f"Hillis-Steele scan, serial octree"
                   f"{', point-label conflict pass' if labels is not None else ''}) in {dt:.2f} s on 1 core "
                   f"({'pinned' if pinned else 'unpinned'}) of {os.cpu_count()} x {cpu}"),
    }


def load_traffic(kernel: str, workload: str):
    """HBM bytes per launch from the committed rocprofv3 counter summary."""
    path = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        with open(path) as f:
            data = json.load(f)
        return data.get(workload, {}).get(kernel)
    except (OSError, ValueError):
        return None


def _batch_roofline(sizes, counts, dim: int, batch_ms: float) -> dict:
    """The byte model summed over the instances (their own m and O), moved in
    one graph replay of the whole segmented pipeline (events around it): the
    replay is one unit, so the pipeline stands for the dominant kernel here;
    per-kernel times are in profiles/batch_4096_instances.md."""
    total = 0
    for n, m, O in zip(sizes, counts["m"], counts["octree_size"]):
        total += algorithmic_bytes(int(n), int(m), int(O), dim, 8, 8)["total"]
    gbps = total / (batch_ms * 1e-3) / 1e9
    return {"kernel": "the segmented pipeline of all instances (one graph replay)",
            "bound": "hbm", "achieved": gbps, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
            "frac": gbps / HBM_PEAK_GBPS, "traffic": None, "avg_launch_ms": batch_ms,
            "algorithmic_bytes": int(total)}


def bench_batch(args) -> int:
    """Batched form: `--batch-count` independent 3D point sets (sizes
    log-uniform in [1e3, 1e6], even instances uniform, odd ones clustered;
    seed 5), 21 bits/axis, through one segmented pipeline replayed as a HIP
    graph, against the plain form launched once per instance
    (pgvd_build_octree + finish each).  Every instance's unique-key and octree
    counts are compared between the two, and every 64th instance's full
    output by device digests."""
    import pgvd_amd as P
    from pgvd_amd import workloads as W

    dim, bits = 3, 21
    sizes = W.batch_sizes(args.batch_count, seed=5)
    t0 = time.perf_counter()
    pts = W.batch_points(sizes, seed=5)
    gen_s = time.perf_counter() - t0
    print(f"batch: {sizes.size} instances, {int(sizes.sum())} points (generated in {gen_s:.1f} s)",
          file=sys.stderr, flush=True)
    dev = P.Device(0)
    dpts = dev.upload(pts)
    offs = np.concatenate([[0], np.cumsum(sizes)])
    b = P.Batch(dev, sizes, dim, bits)
    ipt, rows, dbits, waves = b.tune(dpts)
    sample = b.sample_sort()
    tuned = {"sort": "sample sort", "brt_rows": rows} if sample else {
        "sort": "LSD onesweep", "sort_ipt": ipt, "brt_rows": rows, "digit_bits": dbits,
        "sort_waves": waves}
    print(f"batch: tuned {tuned}", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        b.run(dpts)
        b.finish()
    gpu_ms = []
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        b.run(dpts)
        r = b.finish()
        gpu_ms.append(b.last_ms())
    batch_s = (time.perf_counter() - t0) / args.steps
    counts = P.Batch.counts(r)

    # plain form, one build per instance (warm the pools on the largest first)
    big = int(np.argmax(sizes))
    view = P.DeviceBuffer(dev, dpts.ptr + int(offs[big]) * 12, int(sizes[big]) * 12)
    dev.build_octree_async(view, int(sizes[big]), dim, bits)
    dev.build_octree_finish()
    dev.synchronize()
    m_plain = np.zeros(sizes.size, np.int64)
    o_plain = np.zeros(sizes.size, np.int64)
    t0 = time.perf_counter()
    for i, n in enumerate(sizes):
        view = P.DeviceBuffer(dev, dpts.ptr + int(offs[i]) * 12, int(n) * 12)
        dev.build_octree_async(view, int(n), dim, bits)
        rr = dev.build_octree_finish()
        m_plain[i], o_plain[i] = rr.m, rr.octree_size
    plain_s = time.perf_counter() - t0
    print(f"batch: batched {batch_s * 1e3:.1f} ms/batch, per-instance {plain_s * 1e3:.1f} ms",
          file=sys.stderr, flush=True)

    # digests of every 64th instance's full output, batch vs plain
    kb, nbrt = 8, 16
    checked = 0
    mism = []
    for i in range(0, sizes.size, 64):
        n = int(sizes[i])
        view = P.DeviceBuffer(dev, dpts.ptr + int(offs[i]) * 12, n * 12)
        dev.build_octree_async(view, n, dim, bits)
        rr = dev.build_octree_finish()
        m, O = int(rr.m), int(rr.octree_size)
        k0, o0 = int(counts["key_offset"][i]), int(counts["octree_offset"][i])
        pairs = [
            (rr.keys, r.keys + k0 * kb, m * kb),
            (rr.brt, r.brt + k0 * nbrt, (m - 1) * nbrt),
            (rr.parent, r.parent + k0 * 4, (m - 1) * 4),
            (rr.prefix_sums, r.prefix_sums + k0 * 4, m * 4),
            (rr.octree, r.octree + o0 * 36, O * 36),
        ]
        for a, bb, nbytes in pairs:
            if dev.digest(a, nbytes) != dev.digest(bb, nbytes):
                mism.append(i)
                break
        checked += 1
    same_counts = bool(np.array_equal(m_plain, counts["m"]) and
                      np.array_equal(o_plain, counts["octree_size"]))
    total = int(sizes.sum())
    out = {
        "metric": "batched octree build: sorted Morton keys/sec over a 4096-instance uneven batch",
        "value": total / batch_s,
        "unit": "keys/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": batch_s * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u64",
        "data": "synthetic",
        "config": {
            "workload": f"{sizes.size} independent 3D point sets, sizes log-uniform in [1e3,1e6] "
                        f"(seed 5), even instances uniform in [-1,1]^3, odd ones 8 Gaussian "
                        f"clusters; {bits} bits/axis, 63-bit keys; one segmented pipeline "
                        f"replayed as a HIP graph",
            "instances": int(sizes.size), "total_points": total,
            "tuned": tuned,
        },
        "roofline": _batch_roofline(sizes, counts, dim, float(np.median(gpu_ms))),
        "batched_gpu_ms": float(np.median(gpu_ms)),
        "per_instance_ms": plain_s * 1e3,
        "per_instance_keys_per_s": total / plain_s,
        "speedup_vs_per_instance": plain_s / batch_s,
        "bit_exact": {"counts_equal_all_instances": same_counts,
                      "digest_checked_instances": checked, "digest_mismatches": mism},
    }
    b.close()
    dev.close()
    print(json.dumps(out), flush=True)
    return 0 if (same_counts and not mism) else 1


def bench_serve(args) -> int:
    """Served form: a Poisson stream of octree-build requests (mean
    --serve-rate per second for --serve-seconds), each 2D (16 bits/axis,
    32-bit keys) or 3D (21 bits/axis, 63-bit keys) with equal probability,
    sizes log-uniform in [1e4, 4e6] points (seed 6), points in pinned host
    memory; admitted against a 64 GB HBM budget onto --serve-slots contexts
    whose pooled buffers stay on the device.  Latency = completion - arrival.
    Every 50th request is rebuilt alone and compared (m, octree size, octree
    digest)."""
    import pgvd_amd as P

    rng = np.random.default_rng(6)
    t, arrivals = 0.0, []
    while True:
        t += rng.exponential(1.0 / args.serve_rate)
        if t > args.serve_seconds:
            break
        arrivals.append(t)
    count = len(arrivals)
    sizes = np.exp(rng.uniform(np.log(1e4), np.log(4e6), count)).astype(np.int64)
    dims = rng.choice([2, 3], count)
    pool_n, per_dim = 4_000_000, 8
    pools = {}
    for d in (2, 3):
        for k in range(per_dim):
            pa = P.PinnedArray((pool_n, d))
            pa.array[:] = rng.random((pool_n, d), dtype=np.float32) * 2 - 1
            pools[(d, k)] = pa
    reqs = (P.Request * count)()
    for i in range(count):
        d = int(dims[i])
        r = reqs[i]
        r.host_pts = pools[(d, i % per_dim)].ptr
        r.n, r.dim, r.bits, r.arrival_s = int(sizes[i]), d, 16 if d == 2 else 21, arrivals[i]
    budget = 64 << 30
    print(f"serve: {count} requests over {args.serve_seconds} s, {int(sizes.sum())} points",
          file=sys.stderr, flush=True)
    with P.Server(0, slots=args.serve_slots, hbm_budget=budget) as srv:
        # warm the slots' pools with the largest requests of each dimension
        warm = (P.Request * (2 * args.serve_slots))()
        for j in range(len(warm)):
            d = 2 + (j % 2)
            warm[j].host_pts = pools[(d, 0)].ptr
            warm[j].n, warm[j].dim, warm[j].bits, warm[j].arrival_s = pool_n, d, 16 if d == 2 else 21, 0.0
        srv.run(warm)
        st = srv.run(reqs)
    lat = np.array([reqs[i].done_s - reqs[i].arrival_s for i in range(count)])
    wait = np.array([reqs[i].admit_s - reqs[i].arrival_s for i in range(count)])
    bad = [i for i in range(count) if reqs[i].status != 0]
    # alone rebuilds of every 50th request
    dev = P.Device(0)
    mism = []
    checked = 0
    for i in range(0, count, 50):
        r = reqs[i]
        pts = np.array(pools[(r.dim, i % per_dim)].array[: r.n])
        dpts = dev.upload(pts)
        dev.build_octree_async(dpts, r.n, r.dim, r.bits)
        rr = dev.build_octree_finish()
        dg = dev.digest(rr.octree, rr.octree_size * ((1 << r.dim) + 1) * 4)
        if (rr.m, rr.octree_size, dg) != (r.m, r.octree_size, r.octree_digest):
            mism.append(i)
        checked += 1
        dpts.free()
    dev.close()
    for pa in pools.values():
        pa.free()
    total_pts = int(sizes.sum())
    out = {
        "metric": "served octree builds: throughput with p50/p99 latency (Poisson arrivals)",
        "value": count / st.elapsed_s,
        "unit": "requests/s",
        "n_gpus": 1,
        "higher_is_better": True,
        "data": "synthetic",
        "dtype": "u32/u64",
        "config": {
            "workload": f"Poisson arrivals at {args.serve_rate}/s for {args.serve_seconds} s; 2D "
                        f"(16 bits/axis) or 3D (21 bits/axis) with p=1/2; sizes log-uniform in "
                        f"[1e4, 4e6] (seed 6); points uniform in pinned host memory, copied per "
                        f"request; 64 GB HBM budget; {args.serve_slots} slots",
            "requests": count, "total_points": total_pts,
        },
        "offered_requests_per_s": args.serve_rate,
        "points_per_s": total_pts / st.elapsed_s,
        "latency_ms": {"p50": float(np.percentile(lat, 50) * 1e3),
                       "p99": float(np.percentile(lat, 99) * 1e3),
                       "mean": float(lat.mean() * 1e3), "max": float(lat.max() * 1e3)},
        "queue_wait_ms": {"p50": float(np.percentile(wait, 50) * 1e3),
                          "p99": float(np.percentile(wait, 99) * 1e3)},
        "max_in_flight": st.max_in_flight,
        "max_in_flight_GB": st.max_in_flight_bytes / 1e9,
        "failed": bad,
        "alone_vs_mix": {"checked": checked, "mismatches": mism},
    }
    print(json.dumps(out), flush=True)
    return 0 if not bad and not mism else 1


def _morton3(q, bits: int) -> np.ndarray:
    """Morton keys of 3D grid points (bit i of axis k at bit 3i + k)."""
    key = np.zeros(q.shape[0], np.uint64)
    for i in range(bits):
        for k in range(3):
            key |= ((q[:, k].astype(np.uint64) >> np.uint64(i)) & np.uint64(1)) << np.uint64(3 * i + k)
    return key


def bench_findleaf(args) -> int:
    """Batched point location, OctreeUtils::FindLeaf (OctreeUtils.cpp:18-71):
    2^24 uniform 3D grid points (21 bits/axis, seed 7) located in the octree
    of the 2^24-point uniform build; queries and octree already in HBM.  One
    step = one pgvd_find_leaf call over all queries.  Algorithmic bytes per
    call: 12 B in and 20 B out per query (point; parent, octant, data, level,
    status) plus one read of the octree (36 B per node)."""
    import pgvd_amd as P

    dim, bits = 3, 21
    nq = args.n or (1 << 24)
    pts, desc = make_points("uniform", 1 << 24)
    dev = P.Device(0)
    dpts = dev.upload(pts)
    dev.build_octree_async(dpts, pts.shape[0], dim, bits)
    res = dev.build_octree_finish()
    O = int(res.octree_size)
    q = np.random.default_rng(7).integers(0, 1 << bits, (nq, dim), dtype=np.int32)
    if args.query_order == "morton":
        q = q[np.argsort(_morton3(q, bits), kind="stable")]
    dq = dev.upload(q)
    outs = {k: dev.alloc(nq * 4) for k in ("parent", "octant", "data", "level", "status")}
    for _ in range(max(args.warmup, 1)):
        dev.find_leaf_device(dq, nq, dim, bits, res.octree, O, outs)
    dev.timing(True)
    dev.timing_reset()
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        dev.find_leaf_device(dq, nq, dim, bits, res.octree, O, outs)
    dev.synchronize()
    ms_step = (time.perf_counter() - t0) * 1e3 / args.steps
    kms, kcnt = dev.timing_read("find_leaf")
    launch_ms = kms / max(kcnt, 1)
    dev.timing(False)
    got = {k: dev.download(b, np.uint32 if k == "status" else np.int32, nq) for k, b in outs.items()}
    octree = dev.download(res.octree, np.int32, O * ((1 << dim) + 1)).reshape(O, -1)
    levels = np.bincount(got["level"], minlength=bits + 1)
    dev.close()
    abytes = nq * (12 + 20) + O * ((1 << dim) + 1) * 4
    gbps = abytes / (launch_ms * 1e-3) / 1e9
    out = {
        "metric": "octree point location (FindLeaf) queries/sec on the 2^24-point octree",
        "value": nq / (ms_step * 1e-3),
        "unit": "queries/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "i32",
        "data": "synthetic",
        "config": {
            "workload": f"{nq} uniform grid queries (seed 7"
                        f"{', sorted by Morton key' if args.query_order == 'morton' else ''}) "
                        f"in the octree of {desc}, {bits} bits/axis ({O} octree nodes)",
            "query_order": args.query_order,
            "queries": nq, "octree_nodes": O, "dim": dim, "bits": bits,
            "failed_queries": int((got["status"] != 0).sum()),
            "level_histogram": {int(l): int(c) for l, c in enumerate(levels) if c},
        },
        "roofline": {
            "kernel": ("find_leaf_table_kernel + find_leaf_kernel (the octree's cells at depth 7 "
                       "tabulated, then one lane per query: one table read, then one dependent "
                       "node read per level; timed together)"),
            "bound": "hbm",
            "achieved": gbps,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": gbps / HBM_PEAK_GBPS,
            "traffic": load_traffic("find_leaf", "findleaf" if args.query_order == "random"
                                    else "findleaf_morton"),
            "avg_launch_ms": launch_ms,
            "launches": kcnt,
            "algorithmic_bytes": abytes,
        },
    }
    if not args.no_cpu:
        import oracle
        s = min(args.cpu_sample, nq, 1 << 22)
        t0 = time.perf_counter()
        want = oracle.find_leaf(q[:s], bits, octree[:, :-1], octree[:, -1])
        dt = time.perf_counter() - t0
        mism = sum(int((got[k][:s].astype(np.int64) != want[k].astype(np.int64)).sum())
                   for k in want)
        out["cpu_baseline"] = {
            "value": s / dt, "unit": "queries/s", "cores": 1, "kind": "port",
            "sample": f"first {s} queries, serial FindLeaf restatement on 1 core in {dt:.2f} s",
            "mismatches_vs_gpu": mism,
        }
    print(json.dumps(out), flush=True)
    return 0 if out["config"]["failed_queries"] == 0 and \
        out.get("cpu_baseline", {}).get("mismatches_vs_gpu", 0) == 0 else 1


def bench_cellwalk(args) -> int:
    """Batched CellWalk (viewer/Octree2.cpp:265-313): 2^20 2D segments (seed
    8; a uniform in the grid, b within 1/256 of the grid's width of a) walked
    through the quadtree of 2^22 uniform 2D points at 20 bits/axis; segments
    and quadtree already in HBM.  One step = one pgvd_cell_walk call with a
    cell buffer (a walk keeping each segment's first cells, the offset
    scan, the copy to the offsets, a re-walk of longer segments).  Algorithmic bytes:
    16 B in and 8 B of offset out per segment, 20 B out per visited cell."""
    import pgvd_amd as P

    bits, npts = 20, 1 << 22
    nseg = args.n or (1 << 20)
    rng = np.random.default_rng(8)
    pts = (rng.random((npts, 2), dtype=np.float32) * 2 - 1)
    W = 1 << bits
    a = rng.random((nseg, 2)) * (W - 1e-3)
    b = np.clip(a + (rng.random((nseg, 2)) * 2 - 1) * (W / 256), 0, W - 1e-3)
    segs = np.concatenate([a, b], axis=1).astype(np.float32)
    dev = P.Device(0)
    dpts = dev.upload(pts)
    dev.build_octree_async(dpts, npts, 2, bits)
    res = dev.build_octree_finish()
    O = int(res.octree_size)
    dseg = dev.upload(segs)
    doff = dev.alloc(8 * (nseg + 1))
    L = P.lib()
    total = C.c_int64()
    dev._check(L.pgvd_cell_walk(dev.ctx, dseg.ptr, nseg, bits, res.octree, O, doff.ptr, None, 0,
                                C.byref(total), None, None))
    ncell = total.value
    dcell = dev.alloc(20 * ncell)

    def step():
        dev._check(L.pgvd_cell_walk(dev.ctx, dseg.ptr, nseg, bits, res.octree, O, doff.ptr,
                                    dcell.ptr, ncell, C.byref(total), None, None))

    for _ in range(max(args.warmup, 1)):
        step()
    dev.timing(True)
    dev.timing_reset()
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    dev.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.steps
    c_tot, c_cnt = dev.timing_read("cell_walk_count")
    w_tot, w_cnt = dev.timing_read("cell_walk")
    dev.timing(False)
    # one call = the walk that keeps each segment's first cells (stage
    # "cell_walk_count") + the copy and the re-walk of longer segments
    # ("cell_walk"); both timed by HIP events on the call's stream
    w_launch = c_tot / max(c_cnt, 1) + w_tot / max(w_cnt, 1)
    cells = dev.download(dcell, np.int32, 5 * ncell).reshape(-1, 5) if not args.no_cpu else None
    offs = dev.download(doff, np.int64, nseg + 1) if not args.no_cpu else None
    octree = dev.download(res.octree, np.int32, O * 5).reshape(O, 5) if not args.no_cpu else None
    dev.close()
    wbytes = nseg * 24 + ncell * 20
    gbps = wbytes / (w_launch * 1e-3) / 1e9
    out = {
        "metric": "batched cell walks (CellWalk): visited cells/sec, 2^20 segments in a 2^22-point quadtree",
        "value": ncell / (ms * 1e-3),
        "unit": "cells/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32/i32",
        "data": "synthetic",
        "config": {
            "workload": f"{nseg} segments (seed 8, length up to 1/256 of the grid) through the "
                        f"quadtree of {npts} uniform 2D points at {bits} bits/axis ({O} nodes)",
            "segments": nseg, "cells": ncell, "segments_per_s": nseg / (ms * 1e-3),
            "walk_ms": c_tot / max(c_cnt, 1),
            "copy_and_rewalk_ms": w_tot / max(w_cnt, 1),
        },
        "roofline": {
            "kernel": "cell_walk_kernel (one lane per segment: FindLeaf descents and edge "
                      "intersections per visited cell, the first cells kept) + offset scan + "
                      "walk_compact_kernel + re-walk of longer segments, timed together",
            "bound": "hbm",
            "achieved": gbps,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": gbps / HBM_PEAK_GBPS,
            "traffic": load_traffic("cell_walk", "cellwalk"),
            "avg_launch_ms": w_launch,
            "launches": w_cnt,
            "algorithmic_bytes": wbytes,
        },
    }
    if not args.no_cpu:
        import oracle
        s = min(nseg, 1 << 16)
        t0 = time.perf_counter()
        want = oracle.cell_walk(segs[:s], bits, octree[:, :4], octree[:, 4])
        dt = time.perf_counter() - t0
        same = (np.array_equal(want["offsets"], offs[: s + 1]) and
                np.array_equal(want["cells"], cells[: offs[s]]))
        out["cpu_baseline"] = {
            "value": len(want["cells"]) / dt, "unit": "cells/s", "cores": 1, "kind": "port",
            "sample": f"first {s} segments walked by the serial restatement on 1 core in {dt:.2f} s",
            "equal_to_gpu": bool(same),
        }
    print(json.dumps(out), flush=True)
    return 0 if out.get("cpu_baseline", {}).get("equal_to_gpu", True) else 1


def bench_gvd(args) -> int:
    """The GVD refinement (Octree2::build(const Polylines&) with its
    FindMultiCells, viewer/Octree2.cpp:127-190, 430-506): a scene of 10^4
    closed quadrilateral polylines (seed 11, 2 segments a side, neighbours
    about 5e-4 apart; 90,000 vertices), 24 bits/axis, up to 8 builds.  One
    step = one pgvd_gvd_refine call with the vertices in HBM: quantize, then
    per build the octree of the points, every segment's cell walk with the
    multi-cell visitor, and FitBoxes on the cells two polylines share, whose
    samples join the next build; the host reads one count per stage.
    value = polyline segments walked per second (segments x builds)."""
    import pgvd_amd as P
    from pgvd_amd import workloads

    loops = args.n or 10000
    bits, iters = 24, 8
    v, c = workloads.polyline_scene(loops, 2, 11, 0.0005)
    dev = P.Device(0)
    dv = dev.upload(v)
    for _ in range(max(args.warmup, 1)):
        r, hist = dev.gvd_refine_device(dv, c, bits, iters)
    dev.timing(True)
    dev.timing_reset()
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        r, hist = dev.gvd_refine_device(dv, c, bits, iters)
    dev.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.steps
    stages = {}
    for name in ("gvd_walk", "gvd_walk_write", "gvd_multi_cells", "gvd_fit_count", "gvd_fit_write",
                 "bbox", "encode", "msd", "sort_pass", "unique", "brt", "splits_scan", "malformed",
                 "octree"):
        tot, cnt = dev.timing_read(name)
        if cnt:
            stages[name] = {"ms_per_step": tot / args.steps, "launches_per_step": cnt / args.steps,
                            "avg_ms": tot / cnt}
    dev.timing(False)
    nseg, builds = int(r.n_segments), int(r.iterations)
    got = None
    if not args.no_cpu:
        got = dev.gvd_refine(v, c, bits, iters)
    dev.close()
    walk = stages.get("gvd_walk", {"avg_ms": float("nan"), "launches_per_step": 0})
    # the walk that keeps each segment's first cells: 16 B in, 8 B of
    # offset and a 16 B record per kept cell out per segment; the visited cells are
    # not counted here (they are known only per build)
    wbytes = nseg * 24
    gbps = wbytes / (walk["avg_ms"] * 1e-3) / 1e9
    out = {
        "metric": "GVD refinement (Octree2::build with FindMultiCells): polyline segments walked/sec",
        "value": nseg * builds / (ms * 1e-3),
        "unit": "segments/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32/f64/i32",
        "data": "synthetic",
        "config": {
            "workload": f"{loops} closed quadrilateral polylines (seed 11, 2 segments a side, gaps "
                        f"5e-4) = {v.shape[0]} vertices, {nseg} segments, {bits} bits/axis, up to "
                        f"{iters} builds",
            "segments": nseg, "builds": builds, "extra_points_per_build": hist,
            "final_points": int(r.n_qpoints), "final_octree_nodes": int(r.octree_size),
            "stages": stages,
        },
        "roofline": {
            "kernel": "cell_walk_kernel of the multi-cell walks (one lane per segment)",
            "bound": "hbm",
            "achieved": gbps,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": gbps / HBM_PEAK_GBPS,
            "traffic": None,
            "avg_launch_ms": walk["avg_ms"],
            "launches": walk["launches_per_step"] * args.steps,
            "algorithmic_bytes": wbytes,
        },
    }
    if not args.no_cpu:
        import oracle
        t0 = time.perf_counter()
        want = oracle.gvd_refine(v, c, bits, iters)
        dt = time.perf_counter() - t0
        same = (want["extra_per_iteration"] == got["extra_per_iteration"] and
                np.array_equal(want["qpoints"].astype(np.int32), got["qpoints"]) and
                np.array_equal(want["multi"]["extra"], got["extra"]) and
                np.array_equal(want["tree"]["children"], got["children"]) and
                np.array_equal(want["ci"]["labels"], got["ci_labels"]))
        out["cpu_baseline"] = {
            "value": nseg * want["iterations"] / dt, "unit": "segments/s", "cores": 1,
            "kind": "port",
            "sample": f"the whole refinement ({want['iterations']} builds) by the serial "
                      f"restatement on 1 core in {dt:.2f} s",
            "equal_to_gpu": bool(same),
        }
    print(json.dumps(out), flush=True)
    return 0 if out.get("cpu_baseline", {}).get("equal_to_gpu", True) else 1


def bench_text(args) -> int:
    """The octree's text form (operator<< / operator>>, C/OctNode.h:58-98) on
    the device: the octree of the 2^24-point uniform 3D build (21 bits/axis)
    formatted to text in HBM, and that text parsed back to records.  One step
    = one pgvd_octree_format_text call (the metric) and one
    pgvd_octree_parse_text call, each returning once its length or count is
    read back.  Algorithmic bytes: format reads 36 B per node and writes the
    text; parse reads the text and writes 36 B per node."""
    import pgvd_amd as P

    dim, bits = 3, 21
    pts, desc = make_points("uniform", 1 << 24)
    dev = P.Device(0)
    dpts = dev.upload(pts)
    dev.build_octree_async(dpts, pts.shape[0], dim, bits)
    res = dev.build_octree_finish()
    O = int(res.octree_size)
    rec_bytes = O * ((1 << dim) + 1) * 4
    L = P.lib()
    ln, o2 = C.c_int64(), C.c_int64()
    dev._check(L.pgvd_octree_format_text(dev.ctx, res.octree, O, dim, None, 0, C.byref(ln), None))
    nt = ln.value
    tbuf, obuf = dev.alloc(nt), dev.alloc(rec_bytes)

    def fmt():
        dev._check(L.pgvd_octree_format_text(dev.ctx, res.octree, O, dim, tbuf.ptr, nt,
                                             C.byref(ln), None))

    def prs():
        dev._check(L.pgvd_octree_parse_text(dev.ctx, tbuf.ptr, nt, dim, obuf.ptr, O,
                                            C.byref(o2), None))

    for _ in range(max(args.warmup, 1)):
        fmt()
        prs()
    dev.timing(True)
    dev.timing_reset()
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        fmt()
    fmt_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    t0 = time.perf_counter()
    for _ in range(args.steps):
        prs()
    prs_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    f_tot, f_cnt = dev.timing_read("format_text")
    p_tot, p_cnt = dev.timing_read("parse_text")
    dev.timing(False)
    f_launch, p_launch = f_tot / max(f_cnt, 1), p_tot / max(p_cnt, 1)
    same = dev.digest(obuf, rec_bytes) == dev.digest(res.octree, rec_bytes)
    text_host = dev.download(tbuf, np.uint8, nt).tobytes() if not args.no_cpu else None
    octree_host = dev.download(res.octree, np.int32, O * ((1 << dim) + 1)) if not args.no_cpu else None
    dev.close()
    f_bytes, p_bytes = rec_bytes + nt, nt + rec_bytes
    f_gbps = f_bytes / (f_launch * 1e-3) / 1e9
    out = {
        "metric": "octree text form (operator<<) bytes/s formatted, 2^24-point octree",
        "value": nt / (fmt_ms * 1e-3),
        "unit": "bytes/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": fmt_ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "i32/u8",
        "data": "synthetic",
        "config": {
            "workload": f"octree of {desc}, {bits} bits/axis: {O} nodes formatted to {nt} bytes "
                        "of text in HBM, then parsed back",
            "octree_nodes": O, "text_bytes": nt, "parsed_equal_by_digest": bool(same),
        },
        "parse": {"ms_per_step": prs_ms, "bytes_per_s": nt / (prs_ms * 1e-3),
                  "avg_launch_ms": p_launch,
                  "achieved_GBps": p_bytes / (p_launch * 1e-3) / 1e9,
                  "frac": p_bytes / (p_launch * 1e-3) / 1e9 / HBM_PEAK_GBPS,
                  "traffic": load_traffic("parse_text", "octree_text")},
        "roofline": {
            "kernel": "format_text_kernel (256 nodes per workgroup printed into LDS, look-back "
                      "offsets; with its workspace clear)",
            "bound": "hbm",
            "achieved": f_gbps,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": f_gbps / HBM_PEAK_GBPS,
            "traffic": load_traffic("format_text", "octree_text"),
            "avg_launch_ms": f_launch,
            "launches": f_cnt,
            "algorithmic_bytes": f_bytes,
        },
    }
    if not args.no_cpu:
        import oracle
        stride = (1 << dim) + 1
        s = min(O, 1 << 20)
        sub = octree_host[: s * stride]
        t0 = time.perf_counter()
        txt = oracle.octree_format_text(sub, dim)
        dt = time.perf_counter() - t0
        t0 = time.perf_counter()
        back = oracle.octree_parse_text(txt, dim, cap=s)
        dtp = time.perf_counter() - t0
        out["cpu_baseline"] = {
            "value": len(txt) / dt, "unit": "bytes/s", "cores": 1, "kind": "port",
            "sample": f"first {s} nodes formatted by the serial restatement on 1 core in {dt:.2f} s "
                      f"(parse: {len(txt) / dtp:.3g} bytes/s)",
            "gpu_text_equal": bool(text_host == oracle.octree_format_text(
                octree_host.reshape(O, stride), dim)),
            "parse_equal": bool(back is not None and np.array_equal(back.reshape(-1), sub)),
        }
    print(json.dumps(out), flush=True)
    ok = same and out.get("cpu_baseline", {}).get("gpu_text_equal", True)
    return 0 if ok else 1


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="uniform",
                    choices=["uniform", "gauss", "conflict", "batch", "serve", "findleaf",
                             "octree_text", "cellwalk", "gvd"])
    ap.add_argument("--serve-rate", type=float, default=2000.0)
    ap.add_argument("--serve-seconds", type=float, default=3.0)
    ap.add_argument("--serve-slots", type=int, default=4)
    ap.add_argument("--batch-count", type=int, default=4096)
    ap.add_argument("--n", type=int, default=0, help="points (default 2^24; 2^22 for conflict)")
    ap.add_argument("--query-order", choices=["random", "morton"], default="random",
                    help="findleaf: queries as drawn, or sorted by Morton key (a caller "
                         "whose queries are spatially coherent)")
    ap.add_argument("--cpu-sample", type=int, default=1 << 24)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extra", action="store_true",
                    help="uniform workload only: skip the Gaussian and conflict-cell records")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MiB",
                    help="only run the plain copy kernel over MiB mebibytes (5 launches), "
                         "the reference point for HBM byte counters")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for {args.gpus}): the path runs on one "
              "GPU, and its sharding over several is a design, not built.", file=sys.stderr)
        return 2

    import pgvd_amd as P

    if args.workload == "batch":
        return bench_batch(args)
    if args.workload == "serve":
        return bench_serve(args)
    if args.workload == "findleaf":
        return bench_findleaf(args)
    if args.workload == "octree_text":
        return bench_text(args)
    if args.workload == "cellwalk":
        return bench_cellwalk(args)
    if args.workload == "gvd":
        return bench_gvd(args)

    if args.calibrate_copy:
        nbytes = args.calibrate_copy << 20
        dev = P.Device(0)
        a, b = dev.alloc(nbytes), dev.alloc(nbytes)
        dev.timing(True)
        for _ in range(5):
            dev.copy_kernel(b, a, nbytes)
        ms, cnt = dev.timing_read("copy")
        print(json.dumps({"calibration": "copy_kernel", "bytes_read": nbytes,
                          "bytes_written": nbytes, "launches": cnt,
                          "avg_ms": ms / max(cnt, 1),
                          "GBps": 2 * nbytes / (ms / max(cnt, 1) * 1e-3) / 1e9}))
        dev.close()
        return 0

    out = measure_build(P, args.workload, args.n, args.steps, args.warmup, cpu=not args.no_cpu,
                        cpu_sample=args.cpu_sample)
    if args.workload == "uniform" and not args.no_extra:
        # the configurations the headline hides, measured in the same run:
        # the Gaussian mixture (~28% duplicate keys) and the 126-bit
        # conflict-cell build with labels
        extra = {}
        for w in ("gauss", "conflict"):
            r = measure_build(P, w, 0, args.steps, args.warmup, cpu=False, cpu_sample=0)
            extra[w] = {
                "workload": r["config"]["workload"],
                "ms_per_step": r["ms_per_step"],
                "value": r["value"], "unit": "keys/s",
                "unique_keys": r["config"]["unique_keys"],
                "octree_nodes": r["config"]["octree_nodes"],
                "sort": r["config"]["sort"],
                "frac_of_hbm_peak": r["pipeline"]["frac_of_hbm_peak"],
                "counter_GBps": r["pipeline"]["counter_GBps"],
                "dominant_kernel": r["roofline"]["kernel"],
                "dominant_frac": r["roofline"]["frac"],
            }
        out["other_configs"] = extra
    print(json.dumps(out), flush=True)
    return 0


def counter_bytes_per_step(workload: str):
    """HBM bytes one build moves by the committed rocprofv3 counters: the
    per-launch FETCH+WRITE bytes of every kernel times its launches per
    build (profiles/traffic.json), or None when no summary covers it."""
    path = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        with open(path) as f:
            rec = json.load(f).get(workload, {})
    except (OSError, ValueError):
        return None
    per = rec.get("kernels_bytes_per_launch")
    if not per:
        return None
    launches = rec.get("launches_per_build", {})
    return int(sum(v * launches.get(k, 1) for k, v in per.items()))


def measure_build(P, workload: str, n: int, steps: int, warmup: int, cpu: bool,
                  cpu_sample: int) -> dict:
    """One bench record of the whole path on a synthetic workload (uniform,
    gauss or conflict)."""
    conflict = workload == "conflict"
    dim, bits = 3, (42 if conflict else 21)
    n = n or (1 << 22 if conflict else 1 << 24)
    pts, desc = make_points(workload, n)
    labels = make_points.labels if conflict else None
    dev = P.Device(0)
    dpts = dev.upload(pts)
    dlab = dev.upload(labels) if conflict else None

    # (the LSD passes record a span; the bucket and sample sorts do not)
    dev.timing(True, sort_span_only=True)
    dev.timing_reset()
    res = None
    for _ in range(max(warmup, 1)):
        dev.build_octree_async(dpts, n, dim, bits, dlab)
        res = dev.build_octree_finish()
    bucket = dev.timing_read("sort")[1] == 0

    # Timed region.  HIP events cost ~10 us of queue time each, so the only
    # events inside it are one pair per step around the dominant kernel: the
    # octree gather, or the radix-sort passes where they sorted
    # (launched back to back).
    passes = (dim * bits + 7) // 8
    dev.timing(True, sort_span_only=not bucket, gather_only=bucket)
    dev.timing_reset()
    dev.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        dev.build_octree_async(dpts, n, dim, bits, dlab)
    res = dev.build_octree_finish()
    dev.synchronize()
    elapsed = time.perf_counter() - t0
    ms_step = elapsed * 1e3 / steps
    if bucket:
        dom_ms, dom_cnt = dev.timing_read("gather")
        launch_ms, launches = dom_ms / max(dom_cnt, 1), dom_cnt
    else:
        dom_ms, dom_cnt = dev.timing_read("sort")
        launch_ms, launches = dom_ms / max(dom_cnt, 1) / passes, dom_cnt * passes

    # Per-stage breakdown from separate steps with an event pair per stage
    # (these steps are slower by the event overhead and are not the metric).
    dev.timing(True)
    dev.timing_reset()
    prof_steps = 3
    for _ in range(prof_steps):
        dev.build_octree_async(dpts, n, dim, bits, dlab)
    prof = dev.build_octree_finish()
    flagged = None
    if conflict:
        got = dev.fetch(prof)
        flagged = {"conflict_keys": int(got["key_conflict"].sum()),
                   "nodes_with_conflict_octants": int((got["node_conflict"] != 0).sum())}
    stage_ms = {}
    for st in ["prep", "bbox", "encode", "msd", "sort_pass", "unique", "brt", "splits_scan",
               "malformed", "octree"]:
        tot, cnt = dev.timing_read(st)
        stage_ms[st] = (tot, cnt)
    dev.timing(False)

    m, O = int(res.m), int(res.octree_size)
    lb = 4 if conflict else 0
    ab = algorithmic_bytes(n, m, O, dim, int(res.key_bytes), passes, lb)
    dom_key = "gather" if bucket else "sort_pass"
    dom_gbps = ab[dom_key] / (launch_ms * 1e-3) / 1e9
    total_gbps = ab["total"] / (ms_step * 1e-3) / 1e9
    traffic = load_traffic(dom_key, workload)
    counted = counter_bytes_per_step(workload)
    if bucket:
        dom_name = (f"gather_kernel (scan of local splits and octree fill: {m} BRT nodes into "
                    f"{O} octree nodes; algorithmic bytes {ab['gather']})")
    elif conflict:
        dom_name = "onesweep_kernel (one 8-bit radix pass of 2^22 u128 keys with u32 labels)"
    else:
        dom_name = f"onesweep_kernel (one 8-bit radix pass of {n} u64 keys)"

    out = {
        "metric": (METRIC if not conflict else
                   "sorted Morton keys/sec, conflict-cell octree build at 2^22 pts "
                   "(126-bit keys + uint32 labels); % HBM roofline"),
        "value": n / (ms_step * 1e-3),
        "unit": "keys/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u128" if conflict else "u64",
        "data": "synthetic",
        "config": {
            "workload": f"{desc}, {bits} bits/axis, {dim * bits}-bit keys; full path "
                        "points-in-HBM to octree-in-HBM",
            "n_points": n, "dim": dim, "bits": bits, "distribution": workload,
            "unique_keys": m, "octree_nodes": O, "malformed_brt": int(res.malformed),
            "sort": ("bucket sort (2 scatters + in-LDS buckets)" if res.bucket_sort else
                     "sample sort" if bucket else "LSD onesweep"),
            **({"labels": "uint32 loop id per point", "flags": flagged} if conflict else {}),
        },
        "roofline": {
            "kernel": dom_name,
            "bound": "hbm",
            "achieved": dom_gbps,
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": dom_gbps / HBM_PEAK_GBPS,
            "traffic": traffic,
            "avg_launch_ms": launch_ms,
            "launches": launches,
        },
        "pipeline": {
            "algorithmic_bytes": ab["total"],
            "byte_model": {k: v for k, v in ab.items() if k not in ("total", "sort_pass", "gather")},
            "achieved_GBps": total_gbps,
            "frac_of_hbm_peak": total_gbps / HBM_PEAK_GBPS,
            # HBM bytes the kernels actually move (committed counter
            # summary) over the measured step time, beside the model's rate
            "counter_bytes_per_step": counted,
            "counter_GBps": (counted / (ms_step * 1e-3) / 1e9) if counted else None,
            "stage_ms_per_step": {k: v[0] / prof_steps for k, v in stage_ms.items()},
            "stage_note": "separate steps with an event pair around every stage",
        },
    }
    dev.close()
    if cpu:
        out["cpu_baseline"] = cpu_baseline(pts, bits, min(cpu_sample, n), labels)
    return out


if __name__ == "__main__":
    sys.exit(main())
