"""calcGlobalMemNeeded of a deep tree: its arrays, and the larger of
construction's buffers and of one blocking search beside what the library
keeps of them (at most 1/32 of the device's memory), for sizes whose buffers
are kept and for sizes whose are not. No device calls."""
import numpy as np
import pytest

import pst_amd as P


def _bytes(name, n, *args):
    f = getattr(P.lib(), name)
    f.restype = np.ctypeslib.ctypes.c_size_t
    c = np.ctypeslib.ctypes
    f.argtypes = [c.c_size_t if a is n else c.c_int for a in args]
    return f(*args)


@pytest.mark.parametrize("t,i,n", [("f32", "u32", 1000), ("f32", "u32", 1 << 22), ("f64", "u64", 1 << 26),
                                   ("f32", "u32", (1 << 29) + 3), ("f32", "u32", 1 << 30), ("f64", "u64", 1 << 30)])
def test_needed(t, i, n):
    import torch
    total = torch.cuda.mem_get_info()[1] if torch.cuda.is_available() else 288 << 30
    cus = torch.cuda.get_device_properties(0).multi_processor_count if torch.cuda.is_available() else 256
    dt, idt = P.DT[t], P.DT[i]
    construct = _bytes("_ZN3pst19build_scratch_bytesEiim", n, dt, idt, n)
    search = _bytes("_ZN3pst20search_scratch_bytesEmii", n, n, dt, cus) + n * P.point_dtype(t, i).itemsize
    sz = np.dtype(P.NP[t]).itemsize
    isz = np.dtype(P.NP[i]).itemsize
    slots = (1 << n.bit_length()) - 1
    tree = slots * (P.point_dtype(t, i).itemsize + sz + sz + isz)  # records of a point and a med, minima, IDs
    want = tree + max(construct, min(construct, total // 32) + search)
    assert P.StaticPSTGPU.calcGlobalMemNeeded(n, t, i) == want
