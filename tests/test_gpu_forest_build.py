"""Forest construction with a wave per tree (trees of 31 to 511 points) at the
edges of its range: every tree equals the oracle's tree of its chunk, bit for
bit, with and without a partial last tree, for 32- and 64-bit dims, with IDs
that ascend, do not, repeat or are absent, and with duplicate dims (so that
ties go to the ID and then to the index). The arrays written beside the
records (subtree minima, IDs, dim1 ranges) are checked by counting through
the walk and through the stationary passes."""
import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, _check_trees, _forest, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _points(P, n, t, i, seed, ids):
    rng = np.random.default_rng(seed)
    pts = np.zeros(n, P.point_dtype(t, i))
    span = 40 if seed % 2 else 1 << 20  # few distinct values: ties
    pts["dim1"] = rng.integers(-span, span, n)
    pts["dim2"] = rng.integers(-span, span, n)
    if i is not None:
        pts["id"] = np.arange(n) if ids == "ascending" else rng.permutation(n) if ids == "random" else rng.integers(0, 5, n)
    return pts


CASES = [(tpb, n, t, i, ids)
         for tpb, (t, i, ids) in zip((16, 31, 32, 64, 64, 100, 128, 255, 256, 511, 300),
                                     (("f32", "u32", "random"), ("i64", "u64", "ascending"), ("f64", None, ""),
                                      ("f32", "u32", "ascending"), ("f32", "f32", "repeated"), ("i32", "i64", "random"),
                                      ("f32", "u64", "random"), ("f64", "u32", "ascending"), ("i64", "f64", "random"),
                                      ("f64", "u64", "random"), ("f32", "u32", "ascending")))
         for st in ((1 << int(tpb).bit_length()) - 1,) for n in (st, 7 * st, 9 * st + 1, 6 * st - 1)]


@pytest.mark.parametrize("tpb,n,t,i,ids", CASES)
def test_wave_built_forest(torch, P, tpb, n, t, i, ids):  # noqa: F811
    print(f"forest build tpb={tpb} n={n} {t}/{i} {ids}", flush=True)
    pts = _points(P, n, t, i, tpb + n, ids)
    f, keep = _forest(P, pts, t, i, tpb)
    _check_trees(P, f, pts, t, i)
    rng = np.random.default_rng(n)
    qs = np.zeros(520, P.query_dtype(t))
    lo, hi = pts["dim1"].min(), pts["dim1"].max()
    for name in ("min_dim1", "max_dim1", "min_dim2"):
        qs[name] = rng.integers(int(lo) - 2, int(hi) + 3, len(qs))
    qs["max_dim1"] = np.maximum(qs["max_dim1"], qs["min_dim1"])
    qs["kind"] = rng.integers(0, 3, len(qs))
    want = [len(O.brute_force(pts, int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"])) for q in qs]
    for nq in (200, len(qs)):  # the stationary passes, then the walk
        counts = torch.zeros(nq, dtype=torch.int64, device="cuda")
        f.batch_count(P.to_device(qs[:nq]), nq, counts)
        assert counts.cpu().tolist() == want[:nq], nq
    f.close()
