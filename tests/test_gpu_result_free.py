"""Results of blocking searches belong to the caller, who frees them once, by
pst_free: a second free is an error, as the runtime's is, and what the library
allocates and searches afterwards is unharmed by it."""
import ctypes

import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def test_second_free_is_refused(torch, P):  # noqa: F811
    import pst_data as D
    pts = D.interval_points(300_000, seed=9)
    d = P.to_device(pts)
    q = np.array([0.5], np.float32)
    want = np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q[0], q[0])])
    L = P.lib()
    for _ in range(3):
        tr = P.StaticPSTGPU(d, len(pts), "f32", "u32")
        num, ptr = ctypes.c_size_t(), ctypes.c_void_p()
        P._check(L.pst_gpu_two_sided_left_search(tr.h, P.RET_ID, ctypes.byref(num), ctypes.byref(ptr), q.ctypes.data,
                                                 q.ctypes.data))
        assert np.array_equal(np.sort(P._d2h(ptr.value, num.value * 4).view(np.uint32)), want)
        assert L.pst_free(ptr) == 0
        assert L.pst_free(ptr) == 2  # PST_ERR_HIP
        tr.set_level_index(True)
        assert np.array_equal(np.sort(tr.twoSidedLeftSearch(q[0], q[0])), want)
        tr.close()


def test_cached_memory_is_given_back(torch, P):  # noqa: F811
    import pst_data as D
    n = 3_000_000
    pts = D.interval_points(n, seed=8)
    d = P.to_device(pts)
    P.release_cached_memory()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        tr = P.StaticPSTGPU(d, n, "f32", "u32")
        q = np.float32(0.3)
        assert np.array_equal(np.sort(tr.twoSidedLeftSearch(q, q)), np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q, q)]))
        tr.close()
        kept = free0 - torch.cuda.mem_get_info()[0]
        P.release_cached_memory()
        left = free0 - torch.cuda.mem_get_info()[0]
        print(f"kept {kept}, left after the release {left}", flush=True)
        assert kept > 24 * n and left < (8 << 20)


def test_results_freed_by_the_runtime(torch, P):  # noqa: F811
    """hipFree of a result, before or instead of pst_free, and of one that
    pst_free already took: what is allocated afterwards is sound."""
    import pst_data as D
    path = [ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln][0]
    hip = ctypes.CDLL(path)
    L = P.lib()
    pts = D.interval_points(600_000, seed=12)
    d = P.to_device(pts)
    q = np.array([0.25], np.float32)
    want = np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q[0], q[0])])
    tr = P.StaticPSTGPU(d, len(pts), "f32", "u32")

    def search():
        num, ptr = ctypes.c_size_t(), ctypes.c_void_p()
        P._check(L.pst_gpu_two_sided_left_search(tr.h, P.RET_ID, ctypes.byref(num), ctypes.byref(ptr), q.ctypes.data,
                                                 q.ctypes.data))
        assert np.array_equal(np.sort(P._d2h(ptr.value, num.value * 4).view(np.uint32)), want)
        return ptr

    p = search()
    assert hip.hipFree(p) == 0
    assert L.pst_free(p) == 2  # PST_ERR_HIP
    p = search()
    assert L.pst_free(p) == 0
    assert hip.hipFree(p) == 0  # the caller's mistake: it takes the kept block away
    t = torch.full((600_000,), 7, dtype=torch.int32, device="cuda")  # may lie there now
    for _ in range(3):
        p, r = search(), search()
        assert p.value != r.value
        assert L.pst_free(p) == 0 and L.pst_free(r) == 0
    tr2 = P.StaticPSTGPU(d, len(pts), "f32", "u32")
    assert np.array_equal(np.sort(tr2.twoSidedLeftSearch(q[0], q[0])), want)
    P.release_cached_memory()
    assert bool((t == 7).all())
    tr2.close()
    tr.close()
