"""Metacells of 4 x 4 x 4 voxels with 4-byte values take a kernel of their
own: its minima and maxima have to be the ones of a fold over z, then y, then x
that keeps the first of equal values (bit for bit, so also for zeros of either
sign and for NaN), at the edges of its waves and workgroups."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def fold(vol, pick):
    """vol[z, y, x] -> one value per metacell."""
    for axis in (0, 1, 2):
        g = -(-(vol.shape[axis] - 1) // 4)
        last = vol.shape[axis] - 1
        acc = None
        for k in range(5):
            v = np.take(vol, np.minimum(4 * np.arange(g) + k, last), axis=axis)
            acc = v if acc is None else pick(acc, v)
        vol = acc
    return vol.ravel()


def keep_min(a, b):
    return np.where(b < a, b, a)


def keep_max(a, b):
    return np.where(b > a, b, a)


# (x, y, z) vertices: up to 64, 128 and 256 metacells along x and one more,
# ragged last metacells in each direction; 8-byte values keep the general kernel
@pytest.mark.parametrize("dims,t", [((2, 2, 2), "f32"), ((5, 33, 6), "f64"), ((257, 34, 9), "f32"),
                                    ((258, 17, 10), "i64"), ((513, 18, 5), "f32"), ((514, 9, 7), "i32"),
                                    ((1025, 10, 8), "f32"), ((1030, 8, 6), "f64"), ((12, 301, 1639), "f32"),
                                    ((301, 204, 262), "f32")])
def test_metacells_of_four(dims, t):
    import torch
    import pst_amd as P
    rng = np.random.default_rng(sum(dims))
    px, py, pz = dims
    if t[0] == "i":
        vol = rng.integers(-50, 50, (pz, py, px)).astype(O.NP[t])
    else:
        vol = rng.integers(-3, 4, (pz, py, px)).astype(O.NP[t])
        vol[rng.random(vol.shape) < 0.2] = -0.0
        vol[rng.random(vol.shape) < 0.01] = np.nan
        vol[rng.random(vol.shape) < 0.01] = np.inf
    mn, mxv = fold(vol, keep_min), fold(vol, keep_max)
    n, _ = P.calcNumMetacells(dims, (4, 4, 4))
    assert n == len(mn)
    rec = P.point_dtype(t, "u32")
    # records after the last one must stay as they are
    out = torch.full(((n + 16) * rec.itemsize,), 0xA5, dtype=torch.uint8, device="cuda")
    P.form_metacells_into(torch.from_numpy(vol.ravel()).cuda(), dims, (4, 4, 4), out[:n * rec.itemsize], dtype=t,
                          id_dtype="u32")
    torch.cuda.synchronize()
    raw = out.cpu().numpy()
    got = raw[:n * rec.itemsize].view(rec)
    bits = np.dtype("u4" if vol.itemsize == 4 else "u8")
    for f, want in (("dim1", mn), ("dim2", mxv)):
        g, w = np.ascontiguousarray(got[f]), np.ascontiguousarray(want)
        assert np.array_equal(g.view(bits), w.view(bits))
    assert np.array_equal(got["id"], np.arange(n, dtype=np.uint32))
    assert (raw[n * rec.itemsize:] == 0xA5).all()
