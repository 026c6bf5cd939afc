"""Searches through the level index at the edges of what its plan and copy do
per step: tree heights around the five levels a wave loads at once, run lengths
around the search's probes, batches of one, few and many queries (which probe
and cut their copies differently), outputs around the chunk sizes."""
import numpy as np
import pytest

import oracle as O
from test_gpu_level_index import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,n", [("f32", n) for n in (15, 16, 30, 31, 32, 33, 63, 64, 1022, 1023, 1024, 32767, 32768, 70000)]
                         + [("i64", 1023), ("i64", 33000), ("f64", 31), ("f64", 40001), ("i32", 65535)])
def test_plan_edges(torch, P, t, n):  # noqa: F811
    rng = np.random.default_rng(n)
    pts = np.zeros(n, P.point_dtype(t, "u32"))
    pts["dim1"] = rng.integers(0, max(4, n // 3), n)
    pts["dim2"] = pts["dim1"] + rng.integers(0, 50, n)
    pts["id"] = np.arange(n)
    d = P.to_device(pts)
    tr = P.StaticPSTGPU(d, n, t, "u32")
    tr.set_level_index(True)
    hi = int(pts["dim1"].max())
    for nq in (1, 3, 64, 65, 300):
        print(f"plan {t} n={n} nq={nq}", flush=True)
        qs = np.zeros(nq, P.query_dtype(t))
        qs["min_dim1"] = rng.integers(-2, hi + 2, nq)
        qs["max_dim1"] = qs["min_dim1"] + rng.integers(0, hi + 3, nq) // rng.choice([1, 8, 100], nq)
        qs["min_dim2"] = rng.choice([-5, 1, hi // 2, hi + 60], nq) + rng.integers(0, 9, nq)
        qs["kind"] = rng.integers(0, 3, nq)
        want = [np.sort(pts["id"][O.brute_force(pts, int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"])])
                for q in qs]
        cap = sum(len(w) for w in want)
        counts = torch.zeros(nq, dtype=torch.int64, device="cuda")
        offs = torch.zeros(nq + 1, dtype=torch.int64, device="cuda")
        out = torch.full((cap + 8,), -1, dtype=torch.int32, device="cuda")
        dq = P.to_device(qs)
        tr.batch_search(dq, nq, counts, offs, out, cap)
        r = out.cpu().numpy().view(np.uint32)
        assert counts.cpu().tolist() == [len(w) for w in want]
        o = offs.cpu().numpy()
        for k, w in enumerate(want):
            assert np.array_equal(np.sort(r[o[k]:o[k + 1]]), w), k
        assert np.all(r[cap:] == 0xffffffff)
        # the write call's own plan, clipped to caps
        caps = torch.from_numpy(np.maximum(np.diff(o) - 1, 0)).cuda()
        out2 = torch.full_like(out, -1)
        tr.batch_write(dq, nq, offs, out2, caps_d=caps)
        r2 = out2.cpu().numpy().view(np.uint32)
        for k, w in enumerate(want):
            assert np.array_equal(r2[o[k]:o[k + 1]][:-1], r[o[k]:o[k + 1]][:-1]), k
    for q in qs[:4]:
        k = tr.search_into(int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"], out, cap)
        got = np.sort(out[:k].cpu().numpy().view(np.uint32))
        assert np.array_equal(got, np.sort(pts["id"][O.brute_force(pts, int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"])]))
    tr.close()
