"""Closing a tree and dropping its level index while another
stream is being captured (relaxed or thread-local mode) leaves the capture
whole and frees what it should: the captured work replays, and a tree built
afterwards answers."""
import threading

import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["relaxed", "thread_local"])
def test_frees_beside_a_capture(torch, P, mode):  # noqa: F811
    import pst_data as D
    pts = D.interval_points(200_000, seed=4)
    d = P.to_device(pts)
    q = np.float32(0.4)
    want = np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q, q)])
    trees = [P.StaticPSTGPU(d, len(pts), "f32", "u32") for _ in range(3)]
    for tr in trees:
        tr.set_level_index(True)
        assert np.array_equal(np.sort(tr.twoSidedLeftSearch(q, q)), want)
    x = torch.zeros(1000, device="cuda")
    torch.cuda.synchronize()
    failed = []

    def frees():
        try:
            torch.cuda.set_device(0)
            trees[0].close()
            trees[1].set_level_index(False)
            trees[1].close()
        except BaseException as e:  # noqa: BLE001
            failed.append(repr(e))

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        x.add_(1)
        t = threading.Thread(target=frees)
        t.start()
        t.join()
        x.add_(1)
    assert not failed, failed
    for k in range(3):
        g.replay()
        tr = P.StaticPSTGPU(d, len(pts), "f32", "u32")
        assert np.array_equal(np.sort(tr.twoSidedLeftSearch(q, q)), want)
        tr.close()
        torch.cuda.synchronize()
        assert x[0].item() == 2 * (k + 1)
    trees[2].close()
