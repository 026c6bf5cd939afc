"""Walks whose lists and hand-overs lie beside the lines that choose how they
go on: single searches on trees around the size from which the first workgroup
hands on as soon as it is full, batches whose round lists hold about one, two
and three items per wave, and few queries on a tree above 2^21 points, against
brute force."""
import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _points(P, rng, n):
    pts = np.zeros(n, P.point_dtype("f32", "u32"))
    pts["dim1"] = rng.random(n, dtype=np.float32)
    pts["dim2"] = np.minimum(pts["dim1"] + rng.exponential(0.02, n), 1).astype(np.float32)
    pts["id"] = np.arange(n)
    return pts


@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, (1 << 23) + 1])
def test_single_hand_over(torch, P, n):  # noqa: F811
    rng = np.random.default_rng(n)
    pts = _points(P, rng, n)
    tr = P.StaticPSTGPU(P.to_device(pts), n, "f32", "u32")
    out = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    for kind, lo, hi, m2 in ((O.LEFT, 0, 0.5, 0.5), (O.LEFT, 0, 0.9, 0.2), (O.THREE, 0.2, 0.8, 0.5),
                             (O.THREE, 0.4, 0.4001, 0.4), (O.RIGHT, 0.999, 0, 0.99), (O.THREE, -1, 2, -1)):
        print(f"hand over n={n} {kind} {lo} {hi} {m2}", flush=True)
        lo, hi, m2 = (np.float32(v) for v in (lo, hi, m2))
        want = np.sort(pts["id"][O.brute_force(pts, kind, lo, hi, m2)])
        assert tr.search_into(kind, lo, hi, m2, out, n) == len(want)
        assert np.array_equal(np.sort(out[:len(want)].cpu().numpy().view(np.uint32)), want)
    tr.close()


@pytest.mark.parametrize("n,nqs", [(65536, (3000, 4096)), (300_007, (1500, 3000)), (2_100_000, (8, 40))])
def test_batches_beside_the_lines(torch, P, n, nqs):  # noqa: F811
    rng = np.random.default_rng(n)
    pts = _points(P, rng, n)
    tr = P.StaticPSTGPU(P.to_device(pts), n, "f32", "u32")
    s1, s2 = np.sort(pts["dim1"]), np.sort(pts["dim2"])
    for nq in nqs:
        print(f"lists n={n} nq={nq}", flush=True)
        q = np.zeros(nq, P.query_dtype("f32"))
        q["max_dim1"] = q["min_dim2"] = rng.random(nq, dtype=np.float32)
        q["kind"] = P.LEFT
        # stabbing: dim1 <= v <= dim2, and dim1 <= dim2 for every point
        want = np.searchsorted(s1, q["max_dim1"], "right") - np.searchsorted(s2, q["min_dim2"], "left")
        dq = P.to_device(q)
        counts = torch.zeros(nq, dtype=torch.int64, device="cuda")
        offs = torch.zeros(nq + 1, dtype=torch.int64, device="cuda")
        tr.batch_count(dq, nq, counts)
        assert np.array_equal(counts.cpu().numpy(), want)
        out = torch.full((int(want.sum()) + 1,), -1, dtype=torch.int32, device="cuda")
        tr.batch_search(dq, nq, counts, offs, out, int(want.sum()))
        assert np.array_equal(counts.cpu().numpy(), want)
        r = out.cpu().numpy().view(np.uint32)
        assert r[-1] == 0xffffffff
        o = offs.cpu().numpy()
        for k in range(nq):
            ids = r[o[k]:o[k + 1]]
            p = pts[ids]
            assert np.all((p["dim1"] <= q["max_dim1"][k]) & (p["dim2"] >= q["min_dim2"][k]))
            assert len(np.unique(ids)) == len(ids)
    tr.close()
