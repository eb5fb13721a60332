"""The whole path's bucket sort (bucket.hip) through pgvd_build_octree,
against the oracle: every key width (32-, 64- and 128-bit keys), with and
without labels, at sizes that take each level-0 shape (one LDS item, one
scatter, two scatters), on clustered keys, whose crowded buckets go to the
sample sort or, past its limits, to further levels or the LSD passes, and on
runs of equal keys."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

from conftest import assert_tree_equal

import oracle
import pgvd_amd
from pgvd_amd import workloads

pytestmark = pytest.mark.gpu


def _uniform(n, dim, seed):
    rng = np.random.default_rng(seed)
    return rng.random((n, dim), dtype=np.float32) * 2 - 1


def _clusters(n, dim, seed, k=8, sigma=2e-5):
    """k tight Gaussian clusters (many keys share long prefixes, so whole
    top-level buckets exceed one LDS item) plus the box corners."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.8, 0.8, (k, dim))
    pts = c[rng.integers(0, k, n)] + rng.standard_normal((n, dim)) * sigma
    pts = np.clip(pts, -1, 1).astype(np.float32)
    pts[0] = -1.0
    pts[1] = 1.0
    return pts


def _check(dev, pts, bits, labels=None, where="", bucket=True, **kw):
    print(f"bucket case: {where} n={pts.shape[0]} dim={pts.shape[1]} bits={bits} "
          f"labels={labels is not None}", flush=True)
    got = dev.build_octree(pts, bits, labels=labels, **kw)
    want = oracle.build(oracle.quantize(pts, 1 << bits), bits, labels=labels)
    if bucket is not None:
        assert got["bucket_sort"] == int(bucket), where
    assert_tree_equal(got, want, where=where)
    if labels is not None:
        assert np.array_equal(got["key_conflict"], want["key_conflict"]), where
        assert np.array_equal(got["node_conflict"], want["node_conflict"]), where
    return got


# (dim, bits): 32-bit keys (2D 16 bits), 63-bit (3D 21), 126-bit (3D 42)
@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42)])
@pytest.mark.parametrize("n", [1, 2, 9, 2000, 7000, 60_000, 1 << 20])
def test_bucket_uniform_sizes(dev, dim, bits, n):
    _check(dev, _uniform(n, dim, seed=n % 997 + dim), bits, where="uniform")


@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42)])
@pytest.mark.parametrize("n", [50_000, 1 << 20])
def test_bucket_clustered_levels(dev, dim, bits, n):
    """A sixth of the points in tight clusters: their top-level buckets
    exceed one LDS item and go to the sample sort (through the levels:
    test_bucket_past_the_sample_sort)."""
    pts = _uniform(n, dim, seed=n % 991 + dim)
    k = n // 6
    pts[:k] = _clusters(k, dim, seed=7 + dim)
    _check(dev, pts, bits, where="clusters")


@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42)])
def test_bucket_heavy_clusters(dev, dim, bits):
    """Every point in a tight cluster.  Each crowded bucket of 128-bit keys is
    a segment of the sample sort; keys of at most 64 bits, more than a quarter
    of them crowded, are its segments too or go to the LSD passes (32 bits)."""
    pts = _clusters(1 << 20, dim, seed=17 + dim)
    got = _check(dev, pts, bits, where="heavy clusters", bucket=bits * dim > 64)
    assert got["m"] < pts.shape[0] or bits == 42     # duplicates at the coarser grids


def test_no_host_wait_takes_the_lsd_passes(dev):
    for dim, bits in ((2, 16), (3, 21), (3, 42)):
        _check(dev, _uniform(300_000, dim, seed=5), bits, where="no host wait", bucket=False,
               no_host_wait=True)


def test_bucket_equal_runs(dev):
    """Long runs of one point (a segment whose keys are all equal), beside
    a few others, in all three key widths."""
    for dim, bits in ((2, 16), (3, 21), (3, 42)):
        pts = _uniform(300_000, dim, seed=3)
        pts[1000:200_000] = pts[5]
        pts[250_000:260_000] = pts[7]
        # two thirds of the keys equal: narrower keys take another sort whole
        _check(dev, pts, bits, where="equal runs", bucket=bits * dim > 64)


def test_bucket_labels(dev):
    """Labels travel with their keys through every level (unstable among
    equal keys, which no output observes): conflict flags against the
    oracle, on loops whose samples are copied onto other loops."""
    pts, lab = workloads.star_loops(1 << 19, loops=32, seed=12)
    rng = np.random.default_rng(13)
    src = rng.integers(0, pts.shape[0], 20_000)
    dst = rng.integers(0, pts.shape[0], 20_000)
    pts[dst] = pts[src]
    for bits, dim in ((42, 3), (21, 3)):
        # (63-bit keys on loops: the bucket sort or another, by how clustered)
        _check(dev, pts, bits, labels=lab, where=f"labels {bits}", bucket=True if bits == 42 else None)
    p2 = _clusters(200_000, 2, seed=14, k=4, sigma=1e-3)
    l2 = np.random.default_rng(15).integers(0, 5, p2.shape[0]).astype(np.uint32)
    _check(dev, p2, 16, labels=l2, where="labels 2D", bucket=None)


def test_bucket_13_bit_level0(dev):
    """20 M uniform points: 2^13 top-level buckets (the encode kernel's larger
    bucket histogram), against the oracle."""
    _check(dev, _uniform(20_000_000, 3, seed=25), 21, where="2^13 buckets")


@pytest.mark.parametrize("dim,bits,n,spread", [
    (2, 16, 4099, 1 << 16), (2, 20, 1 << 20, 1 << 20), (3, 21, 600001, 1 << 21),
    (3, 10, 200003, 1 << 10), (2, 30, 70001, 300), (3, 21, 50000, 1)])
def test_int32_grid_points_match_radix(dev, dim, bits, n, spread):
    """int32 grid points take the bucket sort as float points do (the sample
    sort where they crowd): the same tree as with the radix passes that
    no_host_wait asks for.  Coordinates past the grid and below zero keep
    their low bits."""
    rng = np.random.default_rng(n)
    q = rng.integers(0, spread, (n, dim)).astype(np.int32)
    q[::1000] -= 1 << min(bits + 1, 30)
    q[7::1000] += 1 << min(bits, 29)
    got = dev.build_octree(q, bits)
    want = dev.build_octree(q, bits, no_host_wait=True)
    assert want["bucket_sort"] == 0
    assert got["bucket_sort"] == (spread == 1 << bits)      # else crowded
    assert_tree_equal(got, want)


@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42)])
@pytest.mark.parametrize("labels", [False, True])
@pytest.mark.parametrize("kind", ["clusters", "runs", "heavy"])
def test_bucket_past_the_sample_sort(dev, dim, bits, labels, kind):
    """The sorts that take over where a bucket is too large for the sample
    sort, at sizes that reach them by a lower limit: the levels (clusters and
    runs of one point, up to a quarter of the keys; 128-bit keys always) and
    the LSD passes (more of them)."""
    n = 300_007
    pts = _uniform(n, dim, seed=31)
    if kind == "clusters":
        pts[:n // 8] = _clusters(n // 8, dim, seed=5, k=4)
    elif kind == "runs":
        pts[1000:40_000] = pts[5]
        pts[250_000:270_000] = pts[7]
    else:
        pts = _clusters(n, dim, seed=6)
        pts[1000:40_000] = pts[5]
    lab = np.random.default_rng(4).integers(0, 3, n).astype(np.uint32) if labels else None
    lsd = kind == "heavy" and bits != 42
    with pgvd_amd.debug_sort_limits(segment_keys=1):
        _check(dev, pts, bits, labels=lab, where=kind, bucket=not lsd)
        assert dev.last_sort() == ("lsd" if lsd else "levels")


@pytest.mark.parametrize("dim,bits,n,crowd,labels,sort", [
    (3, 21, 4_600_001, 1_100_000, False, "levels"), (3, 21, 3_000_001, 1_100_000, True, "lsd"),
    (3, 21, 4_600_001, 1_000_000, False, "sample buckets"),
    (3, 42, 700_001, 640_000, True, "levels"), (3, 42, 700_001, 600_000, True, "sample buckets"),
    (2, 16, 7_000_001, 1_700_000, False, "levels"), (2, 16, 300_001, 200_000, False, "lsd")])
def test_bucket_at_the_sample_sort_limits(dev, dim, bits, n, crowd, labels, sort):
    """One bucket just below and just above the most keys that the sample sort
    takes (1,048,576 of 64 bits, 628,736 of 128, 1,677,312 of 32), in one cluster
    inside a top-level bucket, a tenth of it one repeated point."""
    pts = _uniform(n, dim, seed=41)
    rng = np.random.default_rng(42)
    pts[:crowd] = 0.4 + rng.standard_normal((crowd, dim)).astype(np.float32) * 2e-4
    pts[:crowd // 10] = pts[0]
    pts[-2], pts[-1] = -1.0, 1.0
    lab = rng.integers(0, 3, n).astype(np.uint32) if labels else None
    got = dev.build_octree(pts, bits, labels=lab)
    assert dev.last_sort() == sort
    want = dev.build_octree(pts, bits, labels=lab, no_host_wait=True)
    assert dev.last_sort() == "lsd"
    assert_tree_equal(got, want)
    if labels:
        for f in ("key_conflict", "node_conflict"):
            assert np.array_equal(got[f], want[f]), f


def test_int32_grid_points_take_the_lsd_passes(dev):
    """Clustered int32 grid points whose largest bucket the sample sort does
    not take."""
    rng = np.random.default_rng(8)
    c = (_clusters(200_003, 2, seed=9, sigma=1e-3) * 0.5 + 0.5) * ((1 << 20) - 1)
    for more in (1000, 1_000_000):       # most of the points crowded, and a few of them
        q = np.concatenate([c.astype(np.int32),
                            rng.integers(0, 1 << 20, (more, 2)).astype(np.int32)])
        want = dev.build_octree(q, 20, no_host_wait=True)
        with pgvd_amd.debug_sort_limits(segment_keys=1):
            got = dev.build_octree(q, 20)
        assert dev.last_sort() in ("lsd", "device") and got["bucket_sort"] == 0
        assert_tree_equal(got, want)


def _grid(n, dim, bits, crowded, seed):
    """int32 grid points, spread evenly or half of them in 8 tight clusters."""
    rng = np.random.default_rng(seed)
    q = rng.integers(0, 1 << bits, (n, dim)).astype(np.int32)
    if crowded:
        c = _clusters(n // 2, dim, seed, sigma=1e-3)
        q[:n // 2] = ((c * 0.5 + 0.5) * ((1 << bits) - 1)).astype(np.int32)
    return q


INT32_CASES = [(2, 16, 4000), (2, 16, 100_003), (2, 20, 300_001), (3, 21, 200_003),
               (3, 10, 1 << 17), (3, 30, 50_001), (2, 20, 800_001), (3, 21, 800_001),
               (2, 16, 1_200_001)]


@pytest.mark.parametrize("dim,bits,n", INT32_CASES)
@pytest.mark.parametrize("labels", [False, True])
def test_int32_build_does_not_wait_for_earlier_work(dev, dim, bits, n, labels):
    """An int32 build returns while the stream still waits for work enqueued
    before it (here a host function that this thread lets go afterwards), and
    the device then chooses its sort."""
    hip = C.CDLL("libamdhip64.so")
    gate, late = threading.Event(), []
    fn = C.CFUNCTYPE(None, C.c_void_p)(lambda _: late.append(1) if not gate.wait(20) else None)
    stream = C.c_void_p()
    dev._check(pgvd_amd.lib().pgvd_ctx_stream(dev.ctx, C.byref(stream)))
    for crowded in (False, True):
        q = _grid(n, dim, bits, crowded, seed=n)
        lab = np.random.default_rng(1).integers(0, 3, n).astype(np.uint32) if labels else None
        want = dev.build_octree(q, bits, labels=lab, no_host_wait=True)
        dev.build_octree(q, bits, labels=lab)          # (allocates)
        d, dl = dev.upload(q), dev.upload(lab) if labels else None
        try:
            gate.clear()
            assert hip.hipLaunchHostFunc(stream, fn, None) == 0
            dev.build_octree_async(d, n, dim, bits, dl, quantized_input=True)
            assert not late
            gate.set()
            r = dev.build_octree_finish()
            got = dev.fetch(r)
            assert dev.last_sort() == ("lsd" if bits == 30 else "buckets" if n == 4000 else "device")
            assert_tree_equal(got, want)
            if labels:
                for f in ("key_conflict", "node_conflict"):
                    assert np.array_equal(got[f], want[f]), f
        finally:
            gate.set()
            dev.synchronize()
            d.free()
            if labels:
                dl.free()


@pytest.mark.parametrize("dim,bits,n", INT32_CASES)
def test_int32_build_under_capture(dev, dim, bits, n):
    """An int32 build captured into a graph (its buffers allocated before) and
    replayed on evenly spread and on clustered points, with eager work between:
    every replay leaves the octree of the points that were there."""
    hip = C.CDLL("libamdhip64.so")
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    dev._check(pgvd_amd.lib().pgvd_ctx_stream(dev.ctx, C.byref(stream)))
    sets = [_grid(n, dim, bits, c, seed=n) for c in (False, True)]
    want = [dev.build_octree(q, bits, no_host_wait=True) for q in sets]
    assert not any(w["malformed"] for w in want)   # (finished on the host)
    d = dev.upload(sets[0])
    try:
        for _ in range(2):
            dev.build_octree_async(d, n, dim, bits, quantized_input=True)
            r = dev.build_octree_finish()
        oct_ptr, stride = r.octree, (1 << dim) + 1
        assert hip.hipStreamBeginCapture(stream, 2) == 0      # relaxed mode
        try:
            dev.build_octree_async(d, n, dim, bits, quantized_input=True)
        finally:
            assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        for which in (0, 1, 1, 0, 1):
            dev._check(pgvd_amd.lib().pgvd_memcpy_htod(dev.ctx, d.ptr, sets[which].ctypes.data,
                                                       sets[which].nbytes, None))
            dev.synchronize()
            assert hip.hipGraphLaunch(run, stream) == 0
            dev.synchronize()
            O = want[which]["octree_size"]
            rec = dev.download(oct_ptr, np.int32, O * stride).reshape(O, stride)
            assert np.array_equal(rec[:, :-1], want[which]["children"])
            assert np.array_equal(rec[:, -1], want[which]["leaf"])
    finally:
        if run:
            hip.hipGraphExecDestroy(run)
        if graph:
            hip.hipGraphDestroy(graph)
        d.free()
    assert_tree_equal(dev.build_octree(sets[1], bits), want[1])
