"""Marching cubes and tetrahedra on metacells of at most 4 x 4 x 4 voxels with
lists long enough that a wave takes several entries, more than 64 of them in
the longest: IDs drawn from a small grid, so that the Python restatement of
each metacell, taken once, gives the whole output, bit for bit and in order;
empty and partial metacells, IDs past the grid (which count and write
nothing), and capacities that end the output in the middle of the list."""
import numpy as np
import pytest

import oracle as O
import test_gpu_isosurface as TET
from test_gpu_marching_cubes import P, ref_metacell, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# entries per wave: 2048 waves up to 16384 IDs, 8 each up to 20480 waves, then more
LISTS = [3000, 6145, 16389, 20480 * 8, 20480 * 64, 20480 * 64 + 20481, 20480 * 70 + 7]


@pytest.mark.parametrize("method", ["cubes", "tetrahedra"])
@pytest.mark.parametrize("dims,mc,t", [((10, 9, 9), (4, 4, 4), "f32"), ((9, 8, 6), (3, 4, 2), "f64"),
                                       ((6, 9, 9), (4, 4, 4), "i32")])
def test_long_lists(torch, P, dims, mc, t, method):  # noqa: F811
    rng = np.random.default_rng(sum(dims) + 7 * sum(mc))
    px, py, pz = dims
    vol = np.full((pz, py, px), 5)
    for _ in range(5):  # a few corners below q: most metacells are empty or nearly so
        vol[rng.integers(0, pz), rng.integers(0, py), rng.integers(0, px)] = -3
    vol = vol.astype(O.NP[t])
    if t != "i32":
        vol += rng.random(vol.shape).astype(O.NP[t]) * O.NP[t](0.25)
    q = 1 if t == "i32" else 1.125
    n, _ = P.calcNumMetacells(dims, mc)
    want = [(ref_metacell if method == "cubes" else TET.ref_metacell)(vol, mc, c, q) for c in range(n)]
    counts1 = np.array([len(w) for w in want] + [0], np.int64)  # the last entry: IDs past the grid
    assert counts1.max() > 0 and counts1.min() == 0
    tri1 = torch.from_numpy(np.array([x for w in want for x in w], np.float32).reshape(-1, 9)).cuda()
    c1 = torch.from_numpy(counts1).cuda()
    first1 = torch.cumsum(c1, 0) - c1
    vd = torch.from_numpy(vol.ravel()).cuda()
    for nids in LISTS:
        print(f"long lists {method} {dims} {t} {nids}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(nids)
        ids = torch.randint(0, n + 1, (nids,), generator=g, device="cuda")
        idd = torch.where(ids == n, n + 5, ids).to(torch.int32)
        per = c1[ids]
        counts = torch.full((nids,), -1, dtype=torch.int64, device="cuda")
        P.isosurface_count(vd, dims, mc, idd, nids, q, counts, dtype=t, method=method)
        assert torch.equal(counts, per)
        offs = torch.zeros(nids + 1, dtype=torch.int64, device="cuda")
        offs[1:] = torch.cumsum(per, 0)
        total = int(offs[-1])
        src = torch.repeat_interleave(first1[ids] - offs[:-1], per) + torch.arange(total, device="cuda")
        ref = tri1[src].view(torch.int32)
        for cap in (total, total * 2 // 3 + 1):
            tri = torch.full((total + 1, 9), 7.0, dtype=torch.float32, device="cuda")
            P.isosurface_write(vd, dims, mc, idd, nids, q, offs, tri, cap, dtype=t, method=method)
            assert torch.equal(tri[:cap].view(torch.int32), ref[:cap])
            assert bool((tri[cap:] == 7.0).all())
