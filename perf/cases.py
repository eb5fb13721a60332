"""The framework's work as a user's program has it done, one case per kind of call.

    listed()            the cases that are timed
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the program holds before the call (inputs on the GPU)
    run(state)          one pass through the public entry points, all outputs
    work(case)          bytes the path cannot do without (no floating-point bound)
    tolerance(case)     every output is bit-exact

Kinds of case ("kind"):
    build   points to octree (Device.build_octree_async + _finish): float
            points or int32 grid points, 2D and 3D, 32- to 126-bit keys, with
            or without object labels
    batch   many independent builds of uneven size (Batch.run + finish)
    find    batched point location (Device.find_leaf_device)
    walk    batched cell walks (pgvd_cell_walk)
    gvd     the GVD refinement loop (Device.gvd_refine_device)
    text    an octree written as text and read back (pgvd_octree_format_text,
            pgvd_octree_parse_text)

A case names a scene (where its clusters, loops and polygons are); the seed
draws the samples of it, so that the counts of another seed are close but not
equal.  Outputs whose length depends on the data come in arrays of a size
fixed by the case (_capacity), entries past the count zero.

Every output is an integer, or a float that fixed float32/float64 steps
determine bit for bit, so there is no 64-bit value to compare with and no
exact(): outputs are compared as they are.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

import pgvd_amd as P
from pgvd_amd.workloads import polyline_scene

MAX_POINTS = 1 << 24


def listed() -> list[dict]:
    return [
        # a small quadtree rebuilt interactively: latency only
        dict(name="quad_1k", kind="build", n=1000, dim=2, bits=16, dist="uniform"),
        # the reference's own test size: 65,536 2D points, 32-bit keys
        dict(name="quad_64k", kind="build", n=65536, dim=2, bits=16, dist="uniform"),
        # an ordinary 3D scan: clustered points, a size that fits no tile
        dict(name="oct_clusters_300k", kind="build", n=300007, dim=3, bits=21, dist="clusters"),
        # the headline workload: 2^24 uniform points, 63-bit keys
        dict(name="oct_uniform_16m", kind="build", n=1 << 24, dim=3, bits=21, dist="uniform"),
        # the same size in clusters so tight that ~28% of the keys repeat
        dict(name="oct_tight_16m", kind="build", n=1 << 24, dim=3, bits=21, dist="tight"),
        # labelled curve samples at full resolution: 126-bit keys, conflict flags
        dict(name="oct_loops_4m", kind="build", n=1 << 22, dim=3, bits=42, dist="loops"),
        # points already on the grid, as Kernels::BuildOctree_p takes them
        dict(name="quad_grid_2m", kind="build", n=2000003, dim=2, bits=20, dist="grid"),
        # many small and middle-sized builds at once
        dict(name="batch_384", kind="batch", count=384, lo=1000, hi=1000000, sizes_seed=5),
        # point location in a large octree, queries in no order
        dict(name="find_16m", kind="find", n=1 << 24, queries=1 << 24, dim=3, bits=21,
             sorted=False),
        # polyline segments walked through a quadtree
        dict(name="walk_1m", kind="walk", dim=2, n=1 << 22, segments=1 << 20, bits=20, reach=256),
        # a scene of polylines refined until no two share a cell
        dict(name="gvd_2500", kind="gvd", loops=2500, bits=24, iterations=8),
        # an octree saved as text and loaded again
        dict(name="text_4m", kind="text", n=1 << 22, dim=3, bits=21),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["build"] * 7 + ["batch", "find", "walk", "gvd", "text"])
    if kind == "build":
        dist = rng.choice(["uniform", "uniform", "clusters", "clusters", "tight", "loops", "grid"])
        dim = 3 if dist in ("tight", "loops") else rng.choice([2, 3])
        if dist == "tight":
            bits = 21
        elif dist == "loops":
            bits = rng.choice([21, 42])
        else:
            bits = rng.choice([16, 20, 24] if dim == 2 else [10, 21])
        hi = MAX_POINTS // 4 if dist == "loops" else MAX_POINTS
        return dict(kind=kind, n=_log_int(rng, 1000, hi), dim=dim, bits=bits, dist=dist)
    if kind == "batch":
        lo = _log_int(rng, 1000, 20000)
        return dict(kind=kind, count=_log_int(rng, 16, 384), lo=lo,
                    hi=_log_int(rng, 2 * lo, 400000), sizes_seed=rng.randrange(1 << 16))
    if kind == "find":
        return dict(kind=kind, n=_log_int(rng, 10000, MAX_POINTS),
                    queries=_log_int(rng, 1000, MAX_POINTS), dim=(dim := rng.choice([2, 3])),
                    bits=16 if dim == 2 else 21, sorted=rng.random() < 0.5)
    if kind == "walk":
        return dict(kind=kind, dim=2, n=_log_int(rng, 10000, MAX_POINTS // 4),
                    segments=_log_int(rng, 1000, 1 << 20), bits=20,
                    reach=_log_int(rng, 256, 4096))
    if kind == "gvd":
        return dict(kind=kind, loops=_log_int(rng, 25, 5000), bits=rng.choice([20, 24]),
                    iterations=8)
    return dict(kind=kind, n=_log_int(rng, 1000, 1 << 22), dim=rng.choice([2, 3]), bits=16)


# ---- inputs -----------------------------------------------------------------

SCENE = 20    # the generator of scenes (clusters, loops, polygons), whatever the seed


@functools.lru_cache(maxsize=1)
def _device() -> P.Device:
    """The program's one context: its buffers serve every call.  The program's
    own torch work runs on the context's stream too."""
    dev = P.Device(0)
    stream = C.c_void_p()
    dev._check(P.lib().pgvd_ctx_stream(dev.ctx, C.byref(stream)))
    torch.cuda.set_stream(torch.cuda.ExternalStream(stream.value))
    return dev


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, n: int, dim: int) -> torch.Tensor:
    return torch.rand((n, dim), generator=g, device="cuda") * 2 - 1


def _clusters(g, n: int, dim: int, k: int, lo: float, hi: float, scene: int = SCENE):
    """n samples of the scene's k Gaussian clusters, widths U[lo, hi], clipped
    to [-1, 1]^dim."""
    rng = np.random.default_rng(scene)
    centres = torch.from_numpy(rng.uniform(-0.9, 0.9, (k, dim))).cuda()
    sig = torch.from_numpy(rng.uniform(lo, hi, k)).cuda()
    comp = torch.randint(0, k, (n,), generator=g, device="cuda")
    pts = torch.randn((n, dim), generator=g, device="cuda").double()
    pts = centres[comp] + pts * sig[comp, None]
    return pts.clamp_(-1, 1).float()


def _loops(g, n: int, loops: int = 64, verts: int = 256):
    """n samples along the scene's closed star-shaped loops in random planes,
    equally many per loop and one in each n-th of its length, with the loop's
    number as label (workloads.star_loops on the GPU)."""
    rng = np.random.default_rng(SCENE)

    def rand(*shape):
        return torch.from_numpy(rng.random(shape)).cuda()

    r0 = rand(loops, 1) * 0.25 + 0.05
    waves = (rand(loops, 1) * 6).floor() + 3
    phi = rand(loops, 1) * (2 * math.pi)
    c = (rand(loops, 1, 3) * 2 - 1) * 0.6
    a = torch.nn.functional.normalize(rand(loops, 1, 3) - 0.5, dim=-1)
    b = rand(loops, 1, 3) - 0.5
    b = torch.nn.functional.normalize(b - a * (a * b).sum(-1, keepdim=True), dim=-1)
    t = torch.arange(verts, device="cuda", dtype=torch.float64)[None] * (2 * math.pi / verts)
    r = r0 * (1 + 0.3 * torch.sin(waves * t + phi))
    v = c + (r * torch.cos(t))[..., None] * a + (r * torch.sin(t))[..., None] * b
    w = v.roll(-1, 1)
    seg = (w - v).norm(dim=-1)
    cum = torch.cat([torch.zeros((loops, 1), device="cuda", dtype=torch.float64),
                     seg.cumsum(1)], 1)
    per = -(-n // loops)
    s = torch.rand((loops, per), generator=g, device="cuda", dtype=torch.float64)
    s = (s + torch.arange(per, device="cuda", dtype=torch.float64)) * (cum[:, -1:] / per)
    j = (torch.searchsorted(cum, s, right=True) - 1).clamp_(0, verts - 1)
    f = ((s - cum.gather(1, j)) / seg.gather(1, j))[..., None]
    j3 = j[..., None].expand(-1, -1, 3)
    pts = v.gather(1, j3)
    pts = pts + f * (w.gather(1, j3) - pts)
    lab = torch.arange(loops, device="cuda", dtype=torch.int32)[:, None].expand(-1, per)
    return (pts.reshape(-1, 3)[:n].float().contiguous(), lab.reshape(-1)[:n].contiguous())


def _scene_polylines(g, loops: int):
    """The scene's closed polylines, every loop moved by up to a tenth of the
    gap between neighbours."""
    gap = 0.05 / math.ceil(math.sqrt(loops))
    v, counts = polyline_scene(loops, 2, SCENE, gap)
    move = (torch.rand((loops, 2), generator=g, device="cuda") - 0.5) * (0.2 * gap)
    of = torch.from_numpy(np.repeat(np.arange(loops), counts)).cuda()
    return (torch.from_numpy(v).cuda() + move[of]).contiguous(), counts


def _points(case: dict, g):
    """(points, labels or None) of a build case."""
    n, dim, dist = case["n"], case["dim"], case["dist"]
    if dist == "loops":
        return _loops(g, n)
    if dist == "clusters":
        return _clusters(g, n, dim, 8, 0.01, 0.1), None
    if dist == "tight":
        pts = _clusters(g, n, dim, 32, 5e-6, 5e-5)
        pts[0], pts[1] = -1.0, 1.0     # the box, and with it the grid, is the uniform case's
        return pts, None
    if dist == "grid":
        return torch.randint(0, 1 << case["bits"], (n, dim), generator=g, device="cuda",
                             dtype=torch.int32), None
    return _uniform(g, n, dim), None


# ---- calls ------------------------------------------------------------------

def _buf(t: torch.Tensor) -> P.DeviceBuffer:
    return P.DeviceBuffer(_device(), t.data_ptr(), t.numel() * t.element_size())


class _Range:
    def __init__(self, ptr: int, shape: tuple, typestr: str):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr=typestr,
                                             strides=None, version=2)


@functools.lru_cache(maxsize=512)
def _view(ptr: int, shape: tuple, typestr: str = "<i4") -> torch.Tensor:
    """The library's device memory as a tensor (no copy)."""
    return torch.as_tensor(_Range(ptr, shape, typestr), device="cuda")


@functools.lru_cache(maxsize=512)
def _past(ptr: int, count: int, rows: int, width: int) -> torch.Tensor:
    return _view(ptr + 4 * width * count, ((rows - count) * width,))


def _whole(*parts) -> list[torch.Tensor]:
    """For each (ptr, count, rows, width) the array of rows x width words at
    ptr, its rows past count cleared (one launch for all)."""
    if any(p[1] > p[2] for p in parts):
        raise ValueError("an output outgrew the array chosen for its case")
    past = [_past(*p) for p in parts if p[1] < p[2]]
    if past:
        torch._foreach_zero_(past)
    return [_view(p[0], (p[2],) if p[3] == 1 else p[2:]) for p in parts]


def _build(pts: torch.Tensor, labels, dim: int, bits: int) -> P.OctreeResult:
    dev = _device()
    dev.build_octree_async(_buf(pts), pts.shape[0], dim, bits,
                           _buf(labels) if labels is not None else None,
                           quantized_input=pts.dtype == torch.int32)
    return dev.build_octree_finish()


class _Plan:
    """A batch plan, given back once neither its state nor its outputs are held."""

    def __init__(self, sizes):
        self.batch = P.Batch(_device(), sizes, 3, 21)

    def __del__(self):
        self.batch.close()


def _batch_sizes(case: dict) -> np.ndarray:
    rng = np.random.default_rng(case["sizes_seed"])
    return np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]),
                              case["count"])).astype(np.int64)


def _batch_points(g, sizes) -> torch.Tensor:
    """Every instance's points, one after another: even instances uniform,
    odd ones in 8 clusters of their own."""
    return torch.cat([_uniform(g, int(n), 3) if i % 2 == 0 else
                      _clusters(g, int(n), 3, 8, 0.01, 0.1, SCENE + i)
                      for i, n in enumerate(sizes)])


def _morton_order(q: torch.Tensor, bits: int) -> torch.Tensor:
    key = torch.zeros(q.shape[0], dtype=torch.int64, device="cuda")
    for b in range(bits):
        for k in range(q.shape[1]):
            key |= ((q[:, k].long() >> b) & 1) << (b * q.shape[1] + k)
    return q[key.argsort()].contiguous()


def _octree_of(case: dict, g) -> torch.Tensor:
    """A copy of the octree of n uniform points, as a program that queries it keeps."""
    dim = case["dim"]
    r = _build(_uniform(g, case["n"], dim), None, dim, case["bits"])
    return _view(r.octree, (r.octree_size, (1 << dim) + 1)).clone()


@functools.lru_cache(maxsize=64)
def _capacity_of(key: tuple) -> tuple:
    case, g = dict(key), _gen(SCENE)
    kind = case["kind"]
    if kind == "gvd":
        v, counts = _scene_polylines(g, case["loops"])
        r, _ = _device().gvd_refine_device(_buf(v), counts, case["bits"], case["iterations"])
        return tuple(int(k * 1.1) + 256 for k in (r.n_qpoints, r.octree_size, r.n_extra,
                                                  r.n_boxes))
    if kind == "batch":
        sizes = _batch_sizes(case)
        pts, plan = _batch_points(g, sizes), _Plan(sizes)
        plan.batch.run(_buf(pts))
        return (int(plan.batch.finish().total_octree * 1.005) + 64,)
    pts, labels = _points(dict(case, dist=case.get("dist", "uniform")), g)
    r = _build(pts, labels, case["dim"], case["bits"])
    return (min(case["n"] + 1, int(r.m * 1.01) + 32),
            min(2 * (case["n"] + 1), int(r.octree_size * 1.02) + 96))


def _capacity(case: dict) -> tuple:
    """Rows of the outputs whose length depends on the data: a little over
    what a first call on the scene reported."""
    return _capacity_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


def prepare(case: dict, seed: int) -> dict:
    _device()
    kind, g = case["kind"], _gen(seed)

    def zeros(*shape, dtype=torch.int32):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    if kind == "build":
        pts, labels = _points(case, g)
        return dict(case=case, pts=pts, labels=labels, rows=_capacity(case))
    if kind == "batch":
        sizes = _batch_sizes(case)
        return dict(case=case, pts=_batch_points(g, sizes), plan=_Plan(sizes),
                    rows=_capacity(case))
    if kind == "find":
        oct_, nq = _octree_of(case, g), case["queries"]
        q = torch.randint(0, 1 << case["bits"], (nq, case["dim"]), generator=g, device="cuda",
                          dtype=torch.int32)
        if case["sorted"]:
            q = _morton_order(q, case["bits"])
        outs = {k: zeros(nq) for k in ("parent", "octant", "data", "level", "status")}
        return dict(case=case, octree=oct_, q=q, outs=outs)
    if kind == "walk":
        oct_, n, reach = _octree_of(case, g), case["segments"], case["reach"]
        W = float(1 << case["bits"])
        a = torch.rand((n, 2), generator=g, device="cuda", dtype=torch.float64) * (W - 1e-3)
        d = torch.rand((n, 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        b = (a + d * (W / reach)).clamp_(0, W - 1e-3)
        cells = int(n * (1.2 + 1.6 * math.sqrt(case["n"]) / reach)) + 1024
        return dict(case=case, octree=oct_, segs=torch.cat([a, b], 1).float().contiguous(),
                    offsets=zeros(n + 1, dtype=torch.int64), status=zeros(n),
                    cells=zeros(cells, 5))
    if kind == "gvd":
        v, counts = _scene_polylines(g, case["loops"])
        rq, ro, re, rb = _capacity(case)
        return dict(case=case, verts=v, counts=counts,
                    kept=dict(qpoints=zeros(rq, 2), octree=zeros(ro, 5),
                              intersections=zeros(ro, 40), extra=zeros(re, 2),
                              samples=zeros(re, 2, dtype=torch.float32),
                              origins=zeros(rb, 2, dtype=torch.float32),
                              lengths=zeros(rb, dtype=torch.float32)))
    nodes, nc = _capacity(case)[1], 1 << case["dim"]
    # every node but the root is named once (up to 8 digits), every other
    # octant is "-1 "
    return dict(case=case, octree=_octree_of(case, g), back=zeros(nodes, nc + 1),
                text=zeros(nodes * (3 * nc + 16), dtype=torch.uint8))


def run(state: dict):
    case, dev = state["case"], _device()
    kind, total = case["kind"], C.c_int64()
    if kind == "build":
        dim = case["dim"]
        r = _build(state["pts"], state["labels"], dim, case["bits"])
        m, nodes, kb = r.m, r.octree_size, r.key_bytes
        M, N = state["rows"]
        parts = dict(keys=(r.keys, m, M, kb // 4),
                     brt=(r.brt, m - 1, M - 1, P.BRT_DTYPES[kb].itemsize // 4),
                     parent=(r.parent, m - 1, M - 1, 1), prefix_sums=(r.prefix_sums, m, M, 1),
                     octree=(r.octree, nodes, N, (1 << dim) + 1))
        if r.key_conflict:
            parts.update(key_conflict=(r.key_conflict, (m + 31) // 32, (M + 31) // 32, 1),
                         node_conflict=(r.node_conflict, nodes, N, 1))
        return dict(zip(parts, _whole(*parts.values())))
    if kind == "batch":
        b = state["plan"].batch
        b.run(_buf(state["pts"]))
        r = b.finish()
        c = P.Batch.counts(r)
        N = state["rows"][0]
        octree = torch.as_tensor(_Range(r.octree, (N, 9), "<i4"), device="cuda")
        octree[r.total_octree:].zero_()
        octree.plan = state["plan"]      # the plan owns this memory
        # (keys, BRT records and parents leave unused slots between the
        # instances; the octrees follow one another without gaps)
        return dict(octree=octree, m=c["m"], octree_size=c["octree_size"],
                    octree_offset=c["octree_offset"])
    if kind == "find":
        dev.find_leaf_device(_buf(state["q"]), case["queries"], case["dim"], case["bits"],
                             _buf(state["octree"]), state["octree"].shape[0],
                             {k: _buf(t) for k, t in state["outs"].items()})
        return state["outs"]
    if kind == "walk":
        dev._check(P.lib().pgvd_cell_walk(
            dev.ctx, state["segs"].data_ptr(), case["segments"], case["bits"],
            state["octree"].data_ptr(), state["octree"].shape[0], state["offsets"].data_ptr(),
            state["cells"].data_ptr(), state["cells"].shape[0], C.byref(total),
            state["status"].data_ptr(), None))
        return dict(offsets=state["offsets"], cells=state["cells"], status=state["status"])
    if kind == "gvd":
        r, per_build = dev.gvd_refine_device(_buf(state["verts"]), state["counts"], case["bits"],
                                             case["iterations"])
        # the next refinement reuses the context's arrays: the program keeps copies
        kept = state["kept"]
        for name, ptr, rows in (("qpoints", r.qpoints, r.n_qpoints),
                                ("octree", r.octree, r.octree_size),
                                ("intersections", r.ci, r.octree_size),
                                ("extra", r.extra, r.n_extra), ("samples", r.samples, r.n_extra),
                                ("origins", r.origins, r.n_boxes),
                                ("lengths", r.lengths, r.n_boxes)):
            if rows:
                t = kept[name]
                t[:rows].copy_(_view(ptr, (rows, *t.shape[1:]),
                                     "<f4" if t.dtype == torch.float32 else "<i4"))
        extra_per_build = np.zeros(case["iterations"], np.int64)
        extra_per_build[:len(per_build)] = per_build
        return dict(kept, extra_per_build=extra_per_build)
    dev._check(P.lib().pgvd_octree_format_text(
        dev.ctx, state["octree"].data_ptr(), state["octree"].shape[0], case["dim"],
        state["text"].data_ptr(), state["text"].numel(), C.byref(total), None))
    dev._check(P.lib().pgvd_octree_parse_text(
        dev.ctx, state["text"].data_ptr(), total.value, case["dim"], state["back"].data_ptr(),
        state["back"].shape[0], C.byref(total), None))
    return dict(text=state["text"], octree=state["back"])


# ---- bounds -----------------------------------------------------------------

def _nodes(n: int, dim: int) -> float:
    """Octree nodes of n spread points, measured on the uniform builds."""
    return (0.473 if dim == 3 else 0.722) * n


def _build_bytes(n: float, dim: int, bits: int, m: float, nodes: float, labels: bool) -> float:
    kb = P.key_bytes_for(dim * bits)
    points = n * (4 * dim + (4 if labels else 0))
    tree = m * (kb + P.BRT_DTYPES[kb].itemsize + 4 + 4) + nodes * 4 * ((1 << dim) + 1)
    return points + tree + ((m / 8 + 4 * nodes) if labels else 0)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "build":
        n, dim, bits = case["n"], case["dim"], case["bits"]
        # the tight clusters: 0.72 distinct keys and 0.26 nodes per point
        m, nodes = (0.72 * n, 0.262 * n) if case["dist"] == "tight" else (n, _nodes(n, dim))
        return dict(bytes=_build_bytes(n, dim, bits, m, nodes, case["dist"] == "loops"), flops=0)
    if kind == "batch":
        n = float(_batch_sizes(case).sum())
        return dict(bytes=_build_bytes(n, 3, 21, n, _nodes(n, 3), False), flops=0)
    if kind == "find":
        dim = case["dim"]
        return dict(bytes=case["queries"] * (4 * dim + 20)
                    + _nodes(case["n"], dim) * 4 * ((1 << dim) + 1), flops=0)
    if kind == "walk":
        # cells a segment crosses: its mean extent over the mean cell width
        cells = case["segments"] * (1 + 1.25 * math.sqrt(case["n"]) / case["reach"])
        return dict(bytes=case["segments"] * 28 + cells * 20, flops=0)
    if kind == "gvd":
        # nine vertices a loop, six builds: segments in and, per build, each
        # node's octree record and intersections out
        n = 9.0 * case["loops"]
        return dict(bytes=n * 8 + 6 * (n * 24 + _nodes(n, 2) * (20 + 160)), flops=0)
    rec = 4 * ((1 << case["dim"]) + 1)
    return dict(bytes=_nodes(case["n"], case["dim"]) * 2 * (rec + 33), flops=0)


def tolerance(case: dict):
    return "exact"
