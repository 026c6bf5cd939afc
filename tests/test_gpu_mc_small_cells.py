"""Marching cubes and tetrahedra on metacells of at most 4 x 4 x 4 voxels (a wave holds a
metacell's vertices) against the Python restatements, bit for bit and in order:
grids whose last metacells are partial on every axis, one-voxel-thick grids,
list lengths around the 64 entries a wave takes at a time, repeated and
unordered IDs, a truncating capacity, and volumes with infinities."""
import numpy as np
import pytest

import oracle as O
import test_gpu_isosurface as TET
from test_gpu_marching_cubes import P, ref_metacell, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["cubes", "tetrahedra"])
@pytest.mark.parametrize("dims,mc,t,nids", [
    ((6, 7, 8), (4, 4, 4), "f32", None), ((2, 2, 2), (4, 4, 4), "f32", None), ((21, 2, 9), (4, 4, 4), "f64", None),
    ((9, 9, 9), (4, 3, 2), "f32", None), ((12, 10, 6), (1, 4, 2), "i64", None), ((18, 17, 18), (4, 4, 4), "i32", None),
    ((18, 17, 18), (4, 4, 4), "f32", 1), ((18, 17, 18), (4, 4, 4), "f32", 63), ((18, 17, 18), (4, 4, 4), "f32", 129)])
def test_small_cells(torch, P, dims, mc, t, nids, method):  # noqa: F811
    rng = np.random.default_rng(sum(dims) * 5 + sum(mc))
    px, py, pz = dims
    if t in ("i32", "i64"):
        vol, q = rng.integers(-9, 9, (pz, py, px)).astype(O.NP[t]), 2
    else:
        vol, q = rng.standard_normal((pz, py, px)).astype(O.NP[t]), 0.05
        if method == "cubes":
            vol[rng.random(vol.shape) < 0.01] = np.inf
            vol[rng.random(vol.shape) < 0.01] = -np.inf
    n, _ = P.calcNumMetacells(dims, mc)
    ids = np.arange(n) if nids is None else rng.integers(0, n, nids)
    ids = rng.permutation(ids).astype(np.uint32)
    print(f"small cells {method} {dims} {mc} {t} {len(ids)}", flush=True)
    vd = torch.from_numpy(vol.ravel()).cuda()
    idd = torch.from_numpy(ids.view(np.int32)).cuda()
    counts = torch.zeros(len(ids), dtype=torch.int64, device="cuda")
    P.isosurface_count(vd, dims, mc, idd, len(ids), q, counts, dtype=t, method=method)
    with np.errstate(invalid="ignore"):
        want = [(ref_metacell if method == "cubes" else TET.ref_metacell)(vol, mc, int(c), q) for c in ids]
    assert counts.cpu().tolist() == [len(w) for w in want]
    offs = np.concatenate([[0], np.cumsum([len(w) for w in want])]).astype(np.int64)
    total = int(offs[-1])
    ref = np.array([x for w in want for x in w], np.float32).reshape(-1)
    for cap in (total, total // 2):
        tri = torch.full((total * 9 + 9,), 7.0, dtype=torch.float32, device="cuda")
        P.isosurface_write(vd, dims, mc, idd, len(ids), q, torch.from_numpy(offs).cuda(), tri, cap, dtype=t,
                           method=method)
        got = tri.cpu().numpy()
        assert np.array_equal(got[:cap * 9], ref[:cap * 9], equal_nan=True)
        assert np.all(got[cap * 9:] == 7.0)
