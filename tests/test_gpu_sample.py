"""The sample sort (sample.hip): clustered builds small enough for it, and the
batched form, against the radix passes and the oracle.  Sizes sit at the
edges of its tiles (4096 or 2048 keys), of one LDS sort (8192, 5120, 3072) and
of its range (512 buckets); sets hold repeated keys that outgrow a bucket."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_tree_equal

import oracle
import pgvd_amd

pytestmark = pytest.mark.gpu

FIELDS = ["keys_lo", "keys_hi", "left", "left_leaf", "right_leaf", "lcp_lo", "lcp_hi",
          "lcp_length", "parent", "prefix_sums", "children", "leaf"]
# 512 buckets of 40% of an LDS sort's keys
LIMIT = {4: 512 * 3276, 8: 512 * 2048}


def clustered(n, dim, seed, sigma=0.02, repeats=()):
    """8 Gaussian clusters; each share of `repeats` replaces that share of the
    points by one of them."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.8, 0.8, (8, dim))
    p = c[rng.integers(0, 8, n)] + rng.standard_normal((n, dim)) * sigma
    at = rng.permutation(n)
    lo = 0
    for share in repeats:
        k = int(share * n)
        p[at[lo:lo + k]] = p[at[lo]]
        lo += k
    p = np.clip(p, -1, 1).astype(np.float32)
    p[0], p[-1] = -1.0, 1.0
    return p


@pytest.mark.parametrize("dim,bits,n,sigma,repeats", [
    (3, 21, 20480, 0.02, ()), (3, 21, 20481, 0.02, ()), (3, 21, 300007, 0.02, ()),
    (3, 21, 300007, 1e-5, ()), (3, 21, 262144, 0.02, (0.4, 0.2, 0.05)),
    (3, 21, 100003, 1e-6, (0.3,)), (2, 30, 70001, 0.001, (0.6,)),
    (2, 16, 200003, 0.01, ()), (3, 10, 150001, 0.02, (0.5,)),
    (3, 21, LIMIT[8], 0.01, ()), (3, 21, LIMIT[8] + 1, 0.01, ()),
    (2, 16, LIMIT[4], 0.01, ()),
    # either side of the largest array that is one segment, by key width
    (2, 16, 1 << 16, 0.01, ()), (2, 16, (1 << 16) + 1, 0.01, ()),
    (2, 20, 3 << 17, 1e-4, ()), (2, 20, (3 << 17) + 1, 1e-4, (0.3,)),
    (3, 21, 1 << 19, 1e-4, (0.3,)), (3, 21, LIMIT[8], 1e-4, (0.2,)),
    # keys that repeat some tens of times each: bins of several keys' copies
    (3, 10, 60000, 0.005, ()), (2, 17, 250000, 2e-4, ())])
def test_clustered_builds_match_radix(dev, dim, bits, n, sigma, repeats):
    pts = clustered(n, dim, n + bits, sigma, repeats)
    got = dev.build_octree(pts, bits)
    want = dev.build_octree(pts, bits, no_host_wait=True)     # the radix passes
    assert want["bucket_sort"] == 0
    assert got["bucket_sort"] == 0        # too clustered for it
    assert_tree_equal(got, want, FIELDS, where=f"n={n} repeats={repeats}")
    if n <= 100003:
        assert_tree_equal(got, oracle.build(oracle.quantize(pts, 1 << bits), bits), FIELDS)


@pytest.mark.parametrize("dim,bits,repeats", [(3, 21, ()), (3, 21, (0.3, 0.1)), (2, 16, (0.2,))])
def test_clustered_builds_with_labels(dev, dim, bits, repeats):
    """Labels ride along: the flags of keys that two labels share."""
    pts = clustered(150003, dim, 7, 0.005, repeats)
    labels = np.random.default_rng(5).integers(0, 3, len(pts)).astype(np.uint32)
    got = dev.build_octree(pts, bits, labels=labels)
    want = dev.build_octree(pts, bits, labels=labels, no_host_wait=True)
    assert_tree_equal(got, want, FIELDS)
    for k in ("key_conflict", "node_conflict"):
        assert np.array_equal(got[k], want[k]), k
    if repeats:
        assert got["key_conflict"].any()


@pytest.mark.parametrize("dim,bits,cap,tile", [(3, 21, 5120, 4096), (2, 16, 8192, 4096),
                                               (3, 42, 3072, 2048)])
def test_batch_matches_radix_passes(dev, dim, bits, cap, tile):
    """Instances of one bucket, just past it and of many, uniform, clustered
    and of one repeated point, in one batch: as with the radix passes that
    sort_waves asks for."""
    sizes = [1, 2, 9, tile - 1, tile + 1, cap - 1, cap, cap + 1, 3 * cap, 40000, 40000, 100003]
    parts = []
    for i, n in enumerate(sizes):
        p = (np.random.default_rng(i).random((n, dim), dtype=np.float32) * 2 - 1 if i % 2 else
             clustered(n, dim, i, 0.003, (0.3, 0.2)) if n > 9 else np.zeros((n, dim), np.float32))
        parts.append(p)
    parts[9][:] = 0.25                       # one key, far above a bucket
    parts[9][0] = -1.0
    pts = np.concatenate(parts)
    d = dev.upload(pts)
    try:
        out = []
        for kw in ({}, {"sort_waves": 3}):
            with pgvd_amd.Batch(dev, sizes, dim, bits, **kw) as b:
                for _ in range(2):           # capture, then replay
                    b.run(d)
                    r = b.finish()
                out.append((b.fetch_all(r), r.key_bytes))
        for i in range(len(sizes)):
            got, want = (pgvd_amd.Batch.instance(a, i, kb, dim) for a, kb in out)
            assert_tree_equal(got, want, FIELDS, where=f"instance {i} (n={sizes[i]})")
    finally:
        d.free()


@pytest.mark.parametrize("dim,bits,n,labels", [(3, 21, 1 << 21, False), (3, 21, 1500001, True),
                                               (3, 42, 700001, True), (2, 16, 1800001, False)])
@pytest.mark.parametrize("share,sigma", [(0.1, 1e-3), (0.9, 1e-3), (0.9, 2e-5)])
def test_crowded_buckets_match_radix(dev, dim, bits, n, labels, share, sigma):
    """Arrays too large to be one segment: the bucket sort's crowded buckets,
    some of them of repeated keys, beside its ordinary ones."""
    pts = np.random.default_rng(3).random((n, dim), dtype=np.float32) * 2 - 1
    k = int(share * n)
    pts[:k] = clustered(k, dim, 9, sigma, (0.1, 0.02))
    lab = np.random.default_rng(5).integers(0, 3, n).astype(np.uint32) if labels else None
    got = dev.build_octree(pts, bits, labels=lab)
    want = dev.build_octree(pts, bits, labels=lab, no_host_wait=True)
    assert want["bucket_sort"] == 0
    assert_tree_equal(got, want, FIELDS)
    if labels:
        for f in ("key_conflict", "node_conflict"):
            assert np.array_equal(got[f], want[f]), f


@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42), (2, 20)])
@pytest.mark.parametrize("labels", [False, True])
@pytest.mark.parametrize("n,crowd", [(60000, 60000), (400001, 400001), (700001, 120000)])
def test_oversize_buckets(dev, dim, bits, labels, n, crowd):
    """Buckets that outgrow an LDS sort, which a sample seldom leaves of
    distinct keys: made of ordinary ones by a lower limit, with runs of
    repeated keys among them, of whole arrays and of crowded buckets in either
    buffer."""
    pts = np.random.default_rng(6).random((n, dim), dtype=np.float32) * 2 - 1
    pts[:crowd] = clustered(crowd, dim, 11, 0.002, (0.2, 0.05))
    lab = np.random.default_rng(5).integers(0, 3, n).astype(np.uint32) if labels else None
    with pgvd_amd.debug_sort_limits(item_keys=700):
        got = dev.build_octree(pts, bits, labels=lab)
    sort = dev.last_sort()
    want = dev.build_octree(pts, bits, labels=lab, no_host_wait=True)
    assert "sample" in sort or (dim, bits) == (2, 16) and n == 400001, sort
    assert_tree_equal(got, want, FIELDS)
    if labels:
        for f in ("key_conflict", "node_conflict"):
            assert np.array_equal(got[f], want[f]), f


@pytest.mark.parametrize("dim,bits", [(2, 16), (3, 21), (3, 42)])
def test_batch_oversize_buckets(dev, dim, bits):
    """The same in a batch, of instances with a prepended zero key and without
    (16384 and 32768 points), one of them on the grid's corner."""
    sizes = [16384, 20000, 32768, 40001, 9, 30000]
    parts = [clustered(n, dim, i, 0.003, (0.3, 0.1)) for i, n in enumerate(sizes)]
    parts[5][:10000] = -1.0
    d = dev.upload(np.concatenate(parts))
    try:
        with pgvd_amd.Batch(dev, sizes, dim, bits) as b, \
                pgvd_amd.debug_sort_limits(item_keys=700):
            assert b.sample_sort()
            for _ in range(2):
                b.run(d)
                r = b.finish()
            all_ = b.fetch_all(r)
        for i, p in enumerate(parts):
            assert_tree_equal(pgvd_amd.Batch.instance(all_, i, r.key_bytes, dim),
                              dev.build_octree(p, bits, no_host_wait=True), FIELDS,
                              where=f"instance {i}")
    finally:
        d.free()
