"""The library keeps freed device blocks for requests of the same size: a tree
that takes a closed tree's blocks answers from its own points alone, also when
threads build, search and close trees of the same sizes at once; what is kept
after every tree is closed stays within 1/32 of the device's memory."""
import threading

import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _check(P, pts, tr):
    for q in (np.float32(0.25), np.float32(0.7)):
        got = np.sort(tr.twoSidedLeftSearch(q, q))
        assert np.array_equal(got, np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q, q)]))


def test_rebuilds_reuse_blocks(torch, P):  # noqa: F811
    import pst_data as D
    total = torch.cuda.mem_get_info()[1]
    free0 = torch.cuda.mem_get_info()[0]
    for n, seed in ((70001, 1), (70001, 2), (3_000_000, 3), (70001, 4), (3_000_000, 5)):
        pts = D.interval_points(n, seed=seed)
        d = P.to_device(pts)
        tr = P.StaticPSTGPU(d, n, "f32", "u32")
        _check(P, pts, tr)
        tr.set_level_index(True)
        _check(P, pts, tr)
        tr.close()
        f = P.StaticPSTGPUArr(d, n, 64)
        _check(P, pts, f)
        f.close()
        del d
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = free0 - torch.cuda.mem_get_info()[0]
    print(f"held after all trees closed: {held}", flush=True)
    assert held <= total // 32 + (64 << 20)  # torch's own context data aside


def test_threads_share_the_cache(torch, P):  # noqa: F811
    import pst_data as D
    failed = []

    def work(k):
        try:
            torch.cuda.set_device(0)
            for r in range(4):
                pts = D.interval_points(50_000, seed=100 * k + r)
                d = P.to_device(pts)
                torch.cuda.synchronize()
                s = torch.cuda.Stream()
                tr = P.StaticPSTGPU(d, len(pts), "f32", "u32", stream=s)
                _check(P, pts, tr)
                tr.close()
        except BaseException as e:  # noqa: BLE001
            failed.append((k, repr(e)))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not failed, failed
