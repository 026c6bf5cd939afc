"""Construction against the oracle's tree, bit for bit, where its paths part
and at the edges of its steps: points that sort once by dim1 with (dim2, ID)
carried along (32-bit dims, IDs rising with the index) beside those that rank
first (64-bit types, unordered or repeated IDs, -0); sizes around the LDS
subtree, the 64-value block minima and their upper steps; inputs whose nodes
all come from one end of every segment, so that removed points pile up there;
extreme values; and a tree that reuses another one's construction block."""
import numpy as np
import pytest

import golden_util as G
import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _points(P, t, i, n, shape, ids, seed):
    rng = np.random.default_rng(seed)
    pts = np.zeros(n, P.point_dtype(t, i))
    if shape == "random":
        pts["dim1"], pts["dim2"] = rng.integers(-10**6, 10**6, n), rng.integers(-10**6, 10**6, n)
    elif shape == "rising":  # dim2 grows with dim1: nodes from every segment's right end
        pts["dim1"], pts["dim2"] = np.arange(n), np.arange(n)
    elif shape == "falling":
        pts["dim1"], pts["dim2"] = np.arange(n), -np.arange(n)
    elif shape == "few":
        pts["dim1"], pts["dim2"] = rng.integers(0, 3, n), rng.integers(0, 3, n)
    elif shape == "equal":
        pts["dim1"], pts["dim2"] = 7, 7
    elif shape == "extreme":
        info = np.finfo(O.NP[t]) if t[0] == "f" else np.iinfo(O.NP[t])
        vals = np.array([info.min, info.max, 0, 1] + ([np.inf, -np.inf] if t[0] == "f" else []), O.NP[t])
        pts["dim1"], pts["dim2"] = rng.choice(vals, n), rng.choice(vals, n)
    elif shape == "zeros":  # -0 and +0: the keys are equal, the stored bits are not
        pts["dim1"], pts["dim2"] = rng.choice(np.array([-0.0, 0.0, 1.0], O.NP[t]), n), rng.choice(
            np.array([-0.0, 0.0, 1.0], O.NP[t]), n)
    if i is not None:
        k = np.arange(n)
        pts["id"] = {"index": k, "gaps": 3 * k + 5, "random": rng.permutation(n), "repeated": k // 3,
                     "signed": k - n // 2}[ids]
    return pts


CASES = [("f32", "u32", n, "random", "index") for n in (1, 2, 63, 64, 65, 2047, 2048, 2049, 4095, 4096, 4097, 4159, 8191,
                                                        8192, 8193, 65535, 65536, 262144, 262145, 300001)]
CASES += [(t, i, 70001, shape, ids) for shape in ("random", "rising", "falling", "few", "equal", "extreme")
          for t, i, ids in (("f32", "u32", "gaps"), ("i32", "i32", "signed"), ("f32", "f32", "index"), ("i32", None, ""),
                            ("f64", "u32", "index"), ("f32", "u64", "index"), ("f32", "u32", "random"),
                            ("i32", "u32", "repeated"), ("i64", "i64", "signed"))]
CASES += [("f32", "u32", 5001, "zeros", "index"), ("f64", "u64", 5001, "zeros", "random"), ("f32", None, 5001, "zeros", "")]


@pytest.mark.parametrize("t,i,n,shape,ids", CASES)
def test_build_paths(torch, P, t, i, n, shape, ids):  # noqa: F811
    print(f"build {t}/{i} n={n} {shape} {ids}", flush=True)
    pts = _points(P, t, i, n, shape, ids, n + len(shape))
    d = P.to_device(pts)
    tr = P.StaticPSTGPU(d, n, t, i)
    ex = tr.export_tree()
    ref = O.build(pts, t, i).arrays()
    for k, v in ref.items():
        assert np.array_equal(G.bits_arr(ex[k]), G.bits_arr(v)), k
    # the subtree minima and the ID array, through a counting batch
    rng = np.random.default_rng(1)
    qs = np.zeros(24, P.query_dtype(t))
    for name in ("min_dim1", "max_dim1", "min_dim2"):
        qs[name] = rng.choice(pts["dim1"] if name != "min_dim2" else pts["dim2"], len(qs))
    qs["kind"] = rng.integers(0, 3, len(qs))
    counts = torch.zeros(len(qs), dtype=torch.int64, device="cuda")
    tr.batch_count(P.to_device(qs), len(qs), counts)
    want = [len(O.brute_force(pts, int(q["kind"]), q["min_dim1"], q["max_dim1"], q["min_dim2"])) for q in qs]
    assert counts.cpu().tolist() == want
    tr.close()


def test_nan_is_refused_on_both_paths(torch, P):  # noqa: F811
    for ids in ("index", "random"):
        for name in ("dim1", "dim2"):
            pts = _points(P, "f32", "u32", 9000, "random", ids, 3)
            pts[name][4567] = np.nan
            with pytest.raises(P.PSTError) as e:
                P.StaticPSTGPU(P.to_device(pts), len(pts), "f32", "u32")
            assert e.value.code == 3
