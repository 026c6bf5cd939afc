"""More open trees than there are slots of pinned result words: searches of the
trees without one copy their results and answer the same, walking and through
the level index."""
import numpy as np
import pytest

import oracle as O
from test_gpu_forest import P, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def test_more_trees_than_result_slots(torch, P):  # noqa: F811
    import pst_data as D
    pts = D.interval_points(3000, seed=6)
    d = P.to_device(pts)
    q = np.float32(0.6)
    want = np.sort(pts["id"][O.brute_force(pts, O.LEFT, 0, q, q)])
    trees = [P.StaticPSTGPU(d, len(pts), "f32", "u32") for _ in range(131)]
    for k, tr in enumerate(trees):
        if k % 2:
            tr.set_level_index(True)
        assert np.array_equal(np.sort(tr.twoSidedLeftSearch(q, q)), want), k
    for tr in trees:
        tr.close()
