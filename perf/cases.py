"""Timed cases: the work that programs have this library do, through its
public entry points, from one small search to the largest trees and volumes.

A case is a dict; its "kind" says which path it takes:

search       blocking drop-in searches on a resident tree, results to the host
search_into  blocking searches through the level index into caller buffers
batch_walk   one batch of searches walking the tree
count        one counting batch walking the tree
batch_index  one batch of ID searches through the level index
graph        the same, replayed as a captured HIP graph
build        a deep tree from a point array, and a small counting batch on it
build_index  a deep tree, its level index, and a small batch of ID searches
forest       volume -> metacells -> forest -> a batch of isovalue searches
surface      active metacells -> triangles, marching cubes or tetrahedra
ips          one interval parallel search (a tree-less stabbing filter)

Points are (min, max) intervals: dim1 ~ U[0, 1), dim2 = dim1 + Exp(0.02)
clamped to 1; integer dims are uniform on [0, 2^30) with geometric widths
of mean 2^12. IDs are the points' indices, or a random permutation of them
("ext": external IDs). Volumes are a sum of Gaussians plus noise.

The order of the IDs that a tree walk or an interval parallel search reports
for one query is unspecified. Where such IDs are the result they are used as
programs use a set: as a mask or a count per point. Output buffers are those
a program keeps: of a size that holds what such queries report, zeroed once.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "static-priority-search-tree_amd"))
import pst_amd as P  # noqa: E402

DEV = "cuda:0"
MEAN = 0.02                 # mean width of float intervals
INT_RANGE, INT_MEAN = 1 << 30, 1 << 12
SIZE = {"f32": 4, "f64": 8, "i32": 4, "i64": 8, "u32": 4, "u64": 8}
REAL = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "i64": torch.int64}
BITS = {4: torch.int32, 8: torch.int64}
METACELL = (4, 4, 4)


def listed():
    return [
        # interactive use of the drop-in API: a few blocking searches on a
        # small tree of odd size, where latency and launches count
        dict(name="search_f32_131k", kind="search", t="f32", id="u32", n=131_075, nq=4),
        # interactive use of a large resident tree: one query at a time
        # through the level index into a kept buffer
        dict(name="search_into_f32_67m", kind="search_into", t="f32", id="u32", n=1 << 26, nq=4),
        # the ordinary batch: 256 stabbing queries on 2^20 intervals
        dict(name="batch_walk_f32_1m", kind="batch_walk", t="f32", id="u32", n=1 << 20, nq=256),
        # sizing a large stream of queries before running it
        dict(name="count_f32_67m", kind="count", t="f32", id="u32", n=1 << 26, nq=2048),
        # the largest batches: gigabytes of IDs through the level index
        dict(name="batch_index_f32_67m", kind="batch_index", t="f32", id="u32", n=1 << 26, nq=1024),
        # a captured serving batch: many queries with short and long outputs
        dict(name="graph_i32_33m", kind="graph", t="i32", id="u32", n=1 << 25, nq=8192),
        # small construction, 64-bit dims and external 64-bit IDs, odd size
        dict(name="build_f64_ext_300k", kind="build", t="f64", id="u64", n=300_007, nq=64, ext=True),
        # the largest construction
        dict(name="build_f32_67m", kind="build", t="f32", id="u32", n=1 << 26, nq=64),
        # an ordinary construction, to the state from which batches are served
        dict(name="build_index_f32_8m", kind="build_index", t="f32", id="u32", n=8_000_003, nq=64),
        # a tree-less filter over all intervals
        dict(name="ips_f32_67m", kind="ips", t="f32", id="u32", n=1 << 26),
        # a new volume: 16.7M metacells, their forest, 200 isovalues
        dict(name="forest_1024", kind="forest", nx=1024, ny=1024, nz=1024, tpb=64, nq=200),
        # the surface of one isovalue of that volume
        dict(name="surface_cubes_1024", kind="surface", nx=1024, ny=1024, nz=1024, method="cubes", level=0.2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search", "search_into", "batch_walk", "count", "batch_index", "graph", "build",
                       "build_index", "ips", "forest", "surface"])
    if kind in ("forest", "surface"):
        dims = [_log(rng, 48, 900) for _ in range(3)]
        c = dict(kind=kind, nx=dims[0], ny=dims[1], nz=dims[2])
        if kind == "forest":
            c.update(tpb=rng.choice([32, 64, 128, 256]), nq=_log(rng, 1, 300))
        else:
            c.update(method=rng.choice(["cubes", "tetrahedra"]), level=round(rng.uniform(0.2, 0.7), 3))
            if c["method"] == "tetrahedra":  # 2.5 times the triangles
                c["nz"] = min(c["nz"], 400)
        return c
    # indexed batches draw sizes below the largest listed one's; the others up to it
    n = {"search": (2_000, 1 << 21), "search_into": (1 << 17, 1 << 25), "batch_walk": (1 << 14, 1 << 21),
         "count": (1 << 16, 1 << 26), "batch_index": (1 << 16, 1 << 25), "graph": (1 << 16, 1 << 25),
         "build": (1_000, 1 << 26), "build_index": (10_000, 1 << 24), "ips": (10_000, 1 << 26)}[kind]
    nq = {"search": (2, 8), "search_into": (2, 8), "batch_walk": (8, 1024), "count": (32, 4096),
          "batch_index": (32, 2000), "graph": (256, 8192), "build": (64, 64), "build_index": (64, 64),
          "ips": (1, 1)}[kind]
    t = rng.choice(["f32", "f32", "i32", "f64", "i64"])
    c = dict(kind=kind, t=t, id="u32", n=_log(rng, *n))
    if kind == "ips":
        return c
    c["nq"] = _log(rng, *nq)
    if kind == "batch_walk":
        c["nq"] = min(c["nq"], 1 + (1 << 29) // c["n"])
    if kind in ("build", "build_index", "search") and rng.random() < 0.4:
        c.update(id=rng.choice(["u32", "u64"]), ext=True)
    if kind == "search" and rng.random() < 0.25:
        c.update(points=True)
    return c


# ---------------------------------------------------------------- inputs

def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(seed * 7919 + 13)


def _dims(case, g):
    """dim1 and dim2 of the case's points, on the GPU."""
    n, t = case["n"], case["t"]
    if t in ("f32", "f64"):
        d1 = torch.rand(n, generator=g, device=DEV, dtype=REAL[t])
        w = torch.empty(n, device=DEV, dtype=REAL[t]).exponential_(1 / MEAN, generator=g)
        return d1, w.add_(d1).clamp_(max=1.0)
    d1 = torch.randint(0, INT_RANGE, (n,), generator=g, device=DEV, dtype=REAL[t])
    w = torch.empty(n, device=DEV, dtype=torch.float32).geometric_(1 / INT_MEAN, generator=g)
    return d1, d1 + (w - 1).to(REAL[t])


def _points(case, g):
    """The point array as bytes, in PointStruct layout."""
    rec = P.point_dtype(case["t"], case["id"])
    n, sz, isz = case["n"], SIZE[case["t"]], SIZE[case["id"]]
    d1, d2 = _dims(case, g)
    ids = (torch.randperm(n, generator=g, device=DEV) if case.get("ext") else torch.arange(n, device=DEV)).to(BITS[isz])
    buf = torch.zeros(n, rec.itemsize, dtype=torch.uint8, device=DEV)
    for name, v, s in (("dim1", d1, sz), ("dim2", d2, sz), ("id", ids, isz)):
        at = rec.fields[name][1]
        buf[:, at:at + s] = v.view(torch.uint8).view(n, s)
    return buf.view(-1)


def _queries(case, seed, stabbing=False):
    """Query records (numpy): stabbing queries (dim1 <= q <= dim2) or the mix
    of ordinary batches: 45% stabbing, 5% right searches near the top of the
    range, 50% three-sided with log-uniform widths. Integer queries have the
    widths of the integer workload, outputs from none to about 10^6."""
    nq, t = case["nq"], case["t"]
    r = np.random.default_rng(seed)
    q = np.zeros(nq, P.query_dtype(t))
    at = np.arange(nq)
    frac = (at * 0.6180339887) % 1.0  # the kinds interleaved, the same in every batch
    left, right = (at >= 0, at < 0) if stabbing else (frac < 0.45, (frac >= 0.45) & (frac < 0.5))
    three = ~left & ~right
    x, c = r.random(nq), r.random(nq)
    if t in ("f32", "f64"):
        w = np.exp(r.uniform(math.log(1e-4), math.log(0.5), nq))
        top = 1 - np.minimum(w, 0.05)
        lo, hi, m2 = x, x + w, c
        m2 = np.where(left, x, np.where(right, top, m2))
    else:
        x, c = np.floor(x * INT_RANGE), np.floor(c * INT_RANGE)
        w = np.floor(np.exp(r.uniform(0, math.log(2.0 ** 23), nq)))
        top = INT_RANGE - 1 - w
        lo, hi = x, x + w
        dense = r.random(nq) < 0.5
        m2 = np.where(dense, np.maximum(x - 1, 0), c)
        m2 = np.where(left, np.maximum(x - (0 if stabbing else w), 0), np.where(right, top, m2))
    q["min_dim1"] = np.where(right, top, lo)
    q["max_dim1"] = np.where(left, x, hi)
    q["min_dim2"] = m2
    q["kind"] = np.where(three, P.THREE, np.where(left, P.LEFT, P.RIGHT))
    return q


def _volume(case, seed):
    """A sum of 64 Gaussians (separable, so a matrix product) plus noise, x fastest."""
    g = _gen(seed)
    dims = (case["nx"], case["ny"], case["nz"])
    centre = torch.rand(3, 64, generator=g, device=DEV)
    sigma = 0.02 + 0.13 * torch.rand(64, generator=g, device=DEV)
    amp = 2 * torch.rand(64, generator=g, device=DEV) - 1
    ex, ey, ez = (torch.exp(-(torch.linspace(0, 1, d, device=DEV)[:, None] - centre[a]) ** 2 / (2 * sigma ** 2))
                  for a, d in enumerate(dims))
    vol = torch.randn(dims[0] * dims[1] * dims[2], generator=g, device=DEV).mul_(0.01).view(dims[2], dims[1], dims[0])
    for z in range(0, dims[2], 64):
        vol[z:z + 64] += torch.matmul((ez[z:z + 64, None, :] * ey[None] * amp), ex.t())
    return vol.view(-1)


def _dims3(case):
    return (case["nx"], case["ny"], case["nz"])


def _isovalue(case, vol):
    return float(np.float32(case["level"] * float(vol.max())))


def _active(case, vol, iso):
    """IDs of the metacells whose (min, max) holds the isovalue, in ascending order."""
    v = vol.view(1, 1, *reversed(_dims3(case)))
    pad = [(-(d - 1)) % m for d, m in zip(_dims3(case), METACELL)]
    v = torch.nn.functional.pad(v, (0, pad[0], 0, pad[1], 0, pad[2]), mode="replicate")
    hi = torch.nn.functional.max_pool3d(v, 5, 4)
    lo = -torch.nn.functional.max_pool3d(-v, 5, 4)
    return torch.nonzero(((lo <= iso) & (hi >= iso)).view(-1)).view(-1).to(torch.int32)


def _batch_buffers(s, case):
    s["counts"] = torch.zeros(case["nq"], dtype=torch.int64, device=DEV)
    s["offsets"] = torch.zeros(case["nq"] + 1, dtype=torch.int64, device=DEV)


def _id_buffer(s, case, cap):
    s["cap"] = cap
    s["out"] = torch.zeros(cap, dtype=BITS[SIZE[case["id"]]], device=DEV)


def _room(case):
    """IDs that a buffer for the case's queries holds: what they report on
    average and five standard deviations."""
    dev = 0.06 if case["t"] in ("f32", "f64") else 0.002
    return int(1.1 * _expected(case) + 5 * dev * case["n"] * math.sqrt(case["nq"])) + 64 * case["nq"]


def _triangle_room(case):
    x, y, z = _dims3(case)
    return (20 if case["method"] == "cubes" else 50) * (x * y + y * z + z * x)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": dict(case), "kind": kind}
    if kind in ("forest", "surface"):
        vol = s["vol"] = _volume(case, seed)
        if kind == "surface":
            s["iso"] = _isovalue(case, vol)
            s["ids"] = _active(case, vol, s["iso"])
            s["cap"] = _triangle_room(case)
            s["counts"] = torch.zeros(P.calcNumMetacells(_dims3(case), METACELL)[0], dtype=torch.int64, device=DEV)
            s["offsets"] = torch.zeros(len(s["counts"]) + 1, dtype=torch.int64, device=DEV)
            s["triangles"] = torch.zeros(s["cap"] * 9, dtype=torch.float32, device=DEV)
            return s
        n, _ = P.calcNumMetacells(_dims3(case), METACELL)
        s["n"], nq = n, case["nq"]
        s["cells"] = torch.zeros(n * 3, dtype=torch.int32, device=DEV)
        q = np.zeros(nq, P.query_dtype("f32"))
        v = np.linspace(float(vol.min()), float(vol.max()), nq + 2)[1:-1]
        q["min_dim1"] = q["max_dim1"] = q["min_dim2"] = v
        q["kind"] = P.LEFT
        s["q"] = P.to_device(q, DEV)
        _batch_buffers(s, case)
        share = 0.02 + 8 / min(_dims3(case))  # of a value range, that a metacell spans
        _id_buffer(s, dict(id="u32"), int(n * (1 + nq * min(share, 1))))
        return s
    g = _gen(seed)
    n, t, i = case["n"], case["t"], case["id"]
    pts = _points(case, g)
    if kind == "ips":
        s["pts"], s["value"] = pts, float(np.float32(0.1 + 0.8 * np.random.default_rng(seed).random()))
        if t not in ("f32", "f64"):
            s["value"] = int(s["value"] * INT_RANGE)
        s["out"] = torch.zeros(n, dtype=torch.int32, device=DEV)
        s["mask"] = torch.zeros(n, dtype=torch.bool, device=DEV)
        s["found"] = torch.zeros(1, dtype=torch.int64, device=DEV)
        return s
    q = s["hq"] = _queries(case, seed, stabbing=kind == "batch_walk")
    s["q"] = P.to_device(q, DEV)
    _batch_buffers(s, case)
    if kind == "search_into":
        s["outs"] = [torch.zeros(n, dtype=BITS[SIZE[i]], device=DEV) for _ in range(case["nq"])]
    elif kind in ("batch_index", "graph", "batch_walk", "build_index"):
        _id_buffer(s, case, _room(case))
    if kind in ("build", "build_index"):
        s["pts"] = pts
        return s
    tree = s["tree"] = P.StaticPSTGPU(pts, n, t, i)
    if kind == "batch_walk":
        s["ones"] = torch.ones(s["cap"], dtype=torch.int32, device=DEV)
    if kind in ("search_into", "batch_index", "graph"):
        tree.set_level_index(True)
    if kind == "graph":
        s["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
        s["graph"] = tree.batch_graph(s["q"], case["nq"], s["counts"], s["offsets"], s["out"], s["cap"], s["stream"])
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    return globals()["_run_" + s["kind"]](s, s["case"])


def _run_search(s, case):
    tree, n, out = s["tree"], case["n"], []
    for q in s["hq"]:
        kind, lo, hi, m2 = int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"]
        mask = np.zeros(n, np.uint8)
        if case.get("points"):
            r = tree.search(kind, lo, hi, m2, ret=P.RET_POINT)
            mask[r["id"]] = 1
            upper = np.zeros(n, r["dim2"].dtype)
            upper[r["id"]] = r["dim2"]
            out.append([mask, upper])
        else:
            mask[tree.search(kind, lo, hi, m2)] = 1
            out.append(mask)
    return out


def _run_search_into(s, case):
    found = []
    for q, buf in zip(s["hq"], s["outs"]):
        found.append(s["tree"].search_into(int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"], buf, len(buf)))
    return [found, s["outs"]]


def _run_batch_walk(s, case):
    # how many of the queries each point answers: the ID sets, counted per point
    s["tree"].batch_search(s["q"], case["nq"], s["counts"], s["offsets"], s["out"], s["cap"])
    total = int(s["offsets"][case["nq"]])
    hits = torch.zeros(case["n"], dtype=torch.int32, device=DEV)
    hits.index_add_(0, s["out"][:total], s["ones"][:total])
    return {"counts": s["counts"], "offsets": s["offsets"], "hits": hits}


def _run_count(s, case):
    s["tree"].batch_count(s["q"], case["nq"], s["counts"])
    return s["counts"]


def _run_batch_index(s, case):
    s["tree"].batch_search(s["q"], case["nq"], s["counts"], s["offsets"], s["out"], s["cap"])
    return {"counts": s["counts"], "offsets": s["offsets"], "ids": s["out"]}


def _run_graph(s, case):
    s["stream"].wait_stream(torch.cuda.current_stream())
    s["graph"].launch(s["stream"])
    torch.cuda.current_stream().wait_stream(s["stream"])
    return {"counts": s["counts"], "offsets": s["offsets"], "ids": s["out"]}


def _run_build(s, case):
    tree = P.StaticPSTGPU(s["pts"], case["n"], case["t"], case["id"])
    tree.batch_count(s["q"], case["nq"], s["counts"])
    tree.close()
    return s["counts"]


def _run_build_index(s, case):
    tree = P.StaticPSTGPU(s["pts"], case["n"], case["t"], case["id"])
    tree.set_level_index(True)
    tree.batch_search(s["q"], case["nq"], s["counts"], s["offsets"], s["out"], s["cap"])
    tree.close()
    return {"counts": s["counts"], "offsets": s["offsets"], "ids": s["out"]}


def _run_ips(s, case):
    # the active intervals as a mask
    P.ips_into(s["pts"], case["n"], s["value"], s["out"], case["n"], s["found"], case["t"], case["id"])
    k = int(s["found"])
    s["mask"].zero_()
    s["mask"][s["out"][:k]] = True
    return {"mask": s["mask"], "found": s["found"]}


def _run_forest(s, case):
    P.form_metacells_into(s["vol"], _dims3(case), METACELL, s["cells"])
    tree = P.StaticPSTGPUArr(s["cells"], s["n"], case["tpb"])
    tree.batch_search(s["q"], case["nq"], s["counts"], s["offsets"], s["out"], s["cap"])
    tree.close()
    return {"cells": s["cells"], "counts": s["counts"], "offsets": s["offsets"], "ids": s["out"]}


def _run_surface(s, case):
    dims, ids, iso, how = _dims3(case), s["ids"], s["iso"], case["method"]
    k = len(ids)
    P.isosurface_count(s["vol"], dims, METACELL, ids, k, iso, s["counts"], method=how)
    torch.cumsum(s["counts"][:k], 0, out=s["offsets"][1:k + 1])
    P.isosurface_write(s["vol"], dims, METACELL, ids, k, iso, s["offsets"], s["triangles"], s["cap"], method=how)
    return {"counts": s["counts"], "triangles": s["triangles"]}


# ---------------------------------------------------------------- exact values

_EDGES = [(0, 1), (2, 3), (4, 5), (6, 7), (0, 2), (1, 3), (4, 6), (5, 7), (0, 4), (1, 5), (2, 6), (3, 7)]
_TETS = [(0, 1, 3, 7), (0, 1, 5, 7), (0, 2, 3, 7), (0, 2, 6, 7), (0, 4, 5, 7), (0, 4, 6, 7)]


def _cube_table():
    """Per configuration (bit k: corner k below), the triangles as edge
    triples: on each face every run of below corners is cut off by a segment
    from the edge where a counter-clockwise walk leaves the run to the edge
    where it entered it; the segments close into loops that are fanned."""
    faces = []
    for a in range(3):
        u, v = 1 << (a + 1) % 3, 1 << (a + 2) % 3
        faces += [[0, v, u | v, u], [1 << a, 1 << a | u, 1 << a | u | v, 1 << a | v]]
    index = {e: k for k, e in enumerate(_EDGES)}
    table = []
    for cfg in range(256):
        step = {}
        for f in faces:
            below = [cfg >> c & 1 for c in f]
            for i in range(4):
                if below[i] and not below[(i + 1) % 4]:
                    j = i
                    while below[j - 1]:
                        j = (j - 1) % 4
                    out, back = (f[i], f[(i + 1) % 4]), (f[j - 1], f[j])
                    step[index[min(out), max(out)]] = index[min(back), max(back)]
        tris, seen = [], set()
        for first in sorted(step):
            loop, e = [], first
            while e not in seen:
                seen.add(e)
                loop.append(e)
                e = step[e]
            tris += [(loop[0], loop[k + 1], loop[k]) for k in range(1, len(loop) - 1)]
        table.append(tris)
    return table


def _voxels(case, ids):
    """Base corners (x, y, z) of the listed metacells' voxels and, for each,
    its metacell's place in the list; x fastest within a metacell."""
    grid = [-(-(d - 1) // m) for d, m in zip(_dims3(case), METACELL)]
    cell = torch.stack([ids % grid[0], ids // grid[0] % grid[1], ids // (grid[0] * grid[1])], 1)
    j = torch.arange(64, device=DEV)
    base = (cell[:, None, :] * 4 + torch.stack([j & 3, j >> 2 & 3, j >> 4], 1)[None]).view(-1, 3)
    inside = (base < torch.tensor([d - 1 for d in _dims3(case)], device=DEV)).all(1)
    owner = torch.arange(len(ids), device=DEV).repeat_interleave(64)
    return base[inside], owner[inside]


_CORNER = torch.tensor([[k & 1, k >> 1 & 1, k >> 2] for k in range(8)])


def _crossing(base, f, iso, u, w):
    """Where the surface crosses the edge between corners u and w (u < w), per voxel."""
    at = torch.arange(len(base), device=DEV)
    corner = _CORNER.to(DEV)
    t = (iso - f[at, u]) / (f[at, w] - f[at, u])
    return base + corner[u] + t[:, None] * (corner[w] - corner[u])


def _exact_cubes(base, owner, f, iso, table, edges):
    cfg = ((f < iso).long() << torch.arange(8, device=DEV)).sum(1)
    number = (table[:, :, 0] >= 0).sum(1)[cfg]
    start = torch.cumsum(number, 0) - number
    tri = torch.empty(int(number.sum()), 9, dtype=torch.float64, device=DEV)
    for k in range(5):
        m = number > k
        e = table[cfg[m], k]
        for c in range(3):
            u, w = edges[e[:, c], 0], edges[e[:, c], 1]
            tri[start[m] + k, 3 * c:3 * c + 3] = _crossing(base[m].double(), f[m], iso, u, w)
    return tri


def _exact_tetrahedra(base, owner, f, iso):
    """In the order metacell, tetrahedron, voxel (a 4x4x4 metacell is one
    chunk of voxels), the second triangle of a quadrilateral after the first."""
    parts, keys = [], []
    at = torch.arange(len(base), device=DEV)
    for n, tet in enumerate(_TETS):
        below = f[:, list(tet)] < iso
        nb = below.sum(1)
        # corners with the below ones first, both halves ascending
        order = torch.tensor(tet, device=DEV)[torch.argsort((~below).long(), dim=1, stable=True)]
        for count, quads in ((1, [((0, 1), (0, 2), (0, 3))]), (3, [((3, 0), (3, 1), (3, 2))]),
                             (2, [((0, 2), (0, 3), (1, 3)), ((0, 2), (1, 3), (1, 2))])):
            m = nb == count
            o, b, g = order[m], base[m].double(), f[m]
            corner = _CORNER.to(DEV).double()
            up = corner[o[:, count]] - corner[o[:, 0]]
            for r, tri in enumerate(quads):
                p = [_crossing(b, g, iso, torch.minimum(o[:, i], o[:, j]), torch.maximum(o[:, i], o[:, j]))
                     for i, j in tri]
                flip = (torch.cross(p[1] - p[0], p[2] - p[0], dim=1) * up).sum(1) < 0
                p1 = torch.where(flip[:, None], p[2], p[1])
                p2 = torch.where(flip[:, None], p[1], p[2])
                parts.append(torch.cat([p[0], p1, p2], 1))
                keys.append(((owner[m] * 6 + n) * len(base) + at[m]) * 2 + r)
    return torch.cat(parts)[torch.argsort(torch.cat(keys))]


def exact(case, seed):
    """Triangles, and the dim2 values of reported points; every other output
    is an integer."""
    if case.get("points"):
        return _exact_points(case, seed)
    if case["kind"] != "surface":
        return None
    vol = _volume(case, seed)
    iso = _isovalue(case, vol)
    ids = _active(case, vol, iso).long()
    v = vol.view(*reversed(_dims3(case)))
    table = torch.full((256, 5, 3), -1, dtype=torch.long)
    for cfg, tris in enumerate(_cube_table()):
        for k, tri in enumerate(tris):
            table[cfg, k] = torch.tensor(tri)
    table, edges = table.to(DEV), torch.tensor(_EDGES, device=DEV)
    parts = []
    for k in range(0, len(ids), 1 << 16):
        base, owner = _voxels(case, ids[k:k + (1 << 16)])
        f = torch.stack([v[base[:, 2] + (c >> 2), base[:, 1] + (c >> 1 & 1), base[:, 0] + (c & 1)]
                         for c in range(8)], 1).double()
        crossed = ((f < iso).sum(1) % 8) != 0
        base, owner, f = base[crossed], owner[crossed], f[crossed]
        parts.append(_exact_cubes(base, owner, f, iso, table, edges) if case["method"] == "cubes"
                     else _exact_tetrahedra(base, owner, f, iso))
    tri = torch.cat(parts) if parts else torch.empty(0, 9, dtype=torch.float64, device=DEV)
    room = torch.zeros(_triangle_room(case) * 9, dtype=torch.float64, device=DEV)
    k = min(tri.numel(), room.numel())
    room[:k] = tri.view(-1)[:k]
    return {"counts": None, "triangles": room}


def _exact_points(case, seed):
    g = _gen(seed)
    d1, d2 = _dims(case, g)
    ids = torch.randperm(case["n"], generator=g, device=DEV) if case.get("ext") else torch.arange(case["n"], device=DEV)
    out = []
    for q in _queries(case, seed):
        kind, lo, hi, m2 = int(q["kind"]), q["min_dim1"].item(), q["max_dim1"].item(), q["min_dim2"].item()
        hit = (d2 >= m2) & ((d1 >= lo) | (kind == P.LEFT)) & ((d1 <= hi) | (kind == P.RIGHT))
        upper = torch.zeros(case["n"], dtype=torch.float64, device=DEV)
        upper[ids[hit]] = d2[hit].double()
        out.append([None, upper])
    return out


# ---------------------------------------------------------------- what a pass cannot do without

def _expected(case):
    """About how many results the case's queries report in all."""
    n, nq = case["n"], case["nq"]
    if case["t"] in ("f32", "f64"):
        stab = MEAN * n
        return nq * stab if case["kind"] == "batch_walk" else nq * (0.45 * stab + 0.05 * 0.005 * n + 0.5 * 0.03 * n)
    stab = n * INT_MEAN / INT_RANGE
    return nq * stab if case["kind"] == "batch_walk" else nq * n * 2.0 ** 23 / 16 / INT_RANGE * 0.75


def work(case):
    kind = case["kind"]
    if kind in ("forest", "surface"):
        vol = 4.0 * case["nx"] * case["ny"] * case["nz"]
        cells = vol / 4 / 64
        if kind == "forest":  # the volume in; metacells and IDs out
            return {"bytes": vol + cells * 12 + 4 * 3.6 * cells * case["nq"] / 200, "flops": 0}
        x, y, z = _dims3(case)  # the active metacells' vertices in, their triangles out
        active = 0.15 * (x * y + y * z + z * x)
        per = 70 if case["method"] == "cubes" else 125
        return {"bytes": active * (64 * 4 + 4 + per * 36), "flops": active * per * 3 * 12}
    n, rec = case["n"], P.point_dtype(case["t"], case["id"]).itemsize
    tree = n * rec
    if kind == "ips":
        return {"bytes": tree + MEAN * n * 4, "flops": 0}
    nq, qb = case["nq"], P.query_dtype(case["t"]).itemsize
    out = _expected(case) * SIZE[case["id"]]
    path = 2 * math.log2(n + 1) * rec * nq  # the boundary paths' nodes
    if kind in ("search", "batch_walk", "search_into", "batch_index", "graph"):
        return {"bytes": nq * (qb + 16) + path + 2 * out * (rec / SIZE[case["id"]] if case.get("points") else 1), "flops": 0}
    if kind == "count":
        return {"bytes": nq * (qb + 8) + path, "flops": 0}
    size = 2.0 ** math.ceil(math.log2(n + 1))
    built = tree + size * (3 * SIZE[case["t"]] + SIZE[case["id"]])
    if kind == "build":
        return {"bytes": built + path, "flops": 0}
    return {"bytes": built + int(n).bit_length() * n * (SIZE[case["t"]] + SIZE[case["id"]]) + path + 2 * out, "flops": 0}
