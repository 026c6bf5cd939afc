"""One search on a deep tree: the workgroup walk that most searches end in, its
hand-over to the round kernels, and its subtree copies in parts, against brute
force: sizes around a full last level (whose subtrees copy as one range) and
beside it (sparse and dense last levels), searches that report next to nothing
and everything, without copies (so that the stack outgrows LDS or the step
bound), with a short copy task list, truncating capacities, points and IDs.
Batches meet the same subtree copies with several queries per walk."""
import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _queries(rng, n, k):
    lo, hi = sorted(rng.integers(0, n, 2))
    return [(O.THREE, -1, n + 1, -1), (O.LEFT, 0, n, n // 2), (O.RIGHT, n // 3, 0, n // 2), (O.THREE, lo, hi, -1),
            (O.THREE, lo, lo + 3, lo), (O.THREE, 5, 2, 0), (O.LEFT, 0, hi, lo)][k]


@pytest.mark.parametrize("t,i,n", [("f32", "u32", n) for n in (1, 2, 3, 511, 4095, 4096, 4700, 8191, 65535, 65536, 65537,
                                                               98304, 131075, 262143, 300007, 1 << 20)]
                         + [("i64", "u64", 100001), ("f64", None, 70000), ("i32", "f32", 131071)])
def test_single_search(torch, P, t, i, n):  # noqa: F811
    rng = np.random.default_rng(n)
    pts = np.zeros(n, P.point_dtype(t, i))
    pts["dim1"], pts["dim2"] = rng.permutation(n), rng.integers(0, n, n)
    if i is not None:
        pts["id"] = np.arange(n)
    tr = P.StaticPSTGPU(P.to_device(pts), n, t, i)
    rec = pts.dtype if i is None else np.dtype(O.NP[i])
    out = torch.full(((n + 4) * rec.itemsize,), 255, dtype=torch.uint8, device="cuda")
    for copies in ((256, 65535, 0), (16, 1 << 20, 0), (0, 0, 0), (16, 65535, 3)):
        tr.set_subtree_copy(*copies)
        for k in range(7):
            kind, lo, hi, m2 = _queries(rng, n, k)
            hit = O.brute_force(pts, kind, lo, hi, m2)
            want = np.sort(pts[hit] if i is None else pts["id"][hit])
            for cap in (n, len(want) // 2):
                print(f"single {t}/{i} n={n} copies={copies} q={k} cap={cap}", flush=True)
                out.fill_(255)
                got = tr.search_into(kind, lo, hi, m2, out, cap)
                assert got == len(want)
                r = out.cpu().numpy().view(rec)
                k2 = min(cap, len(want))
                if k2 == len(want):
                    assert np.array_equal(np.sort(r[:k2]), want)
                else:
                    assert len(np.unique(r[:k2])) == k2 and np.all(np.isin(r[:k2], want))
                assert np.all(r[k2:].view(np.uint8) == 255)
    if i is not None:
        tr.set_subtree_copy(256, 65535, 0)
        kind, lo, hi, m2 = _queries(rng, n, 3)
        got = np.sort(tr.search(kind, lo, hi, m2, ret=P.RET_POINT), order="id")
        assert np.array_equal(got, pts[O.brute_force(pts, kind, lo, hi, m2)])
    tr.close()


@pytest.mark.parametrize("n", [5000, 65536, 70001, 98304, 131073, 200000])
def test_batch_copies_of_ragged_subtrees(torch, P, n):  # noqa: F811
    rng = np.random.default_rng(n)
    pts = np.zeros(n, P.point_dtype("f32", "u32"))
    pts["dim1"], pts["dim2"], pts["id"] = rng.permutation(n), rng.integers(0, n, n), np.arange(n)
    tr = P.StaticPSTGPU(P.to_device(pts), n, "f32", "u32")
    tr.set_subtree_copy(16, 1 << 20, 0)
    qs = np.zeros(37, P.query_dtype("f32"))
    for q in qs:
        kind, lo, hi, m2 = _queries(rng, n, int(rng.integers(0, 7)))
        q["kind"], q["min_dim1"], q["max_dim1"], q["min_dim2"] = kind, lo, hi, m2 if rng.random() < 0.5 else -1
    want = [np.sort(pts["id"][O.brute_force(pts, int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"])]) for q in qs]
    total = sum(len(w) for w in want)
    counts = torch.zeros(len(qs), dtype=torch.int64, device="cuda")
    offs = torch.zeros(len(qs) + 1, dtype=torch.int64, device="cuda")
    out = torch.full((total + 4,), -1, dtype=torch.int32, device="cuda")
    tr.batch_search(P.to_device(qs), len(qs), counts, offs, out, total)
    o, r = offs.cpu().numpy(), out.cpu().numpy().view(np.uint32)
    for k, w in enumerate(want):
        assert np.array_equal(np.sort(r[o[k]:o[k + 1]]), w), k
    assert np.all(r[total:] == 0xffffffff)
    tr.close()
