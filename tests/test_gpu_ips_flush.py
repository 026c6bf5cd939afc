"""The interval search writes what its waves still hold at the end with one
reservation per workgroup, and reads arrays beyond the last-level cache as
streaming: every hit has to be there once, whatever waves hold, up to the
capacity."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# chunks are 1024 points, workgroups four chunks; 0 to all points hit; the
# last size is beyond 256 MB
@pytest.mark.parametrize("n,every", [(1, 1), (63, 2), (1024, 1), (1025, 3), (4096, 5), (4097, 4000), (70001, 1),
                                     (1 << 20, 7), (1 << 20, 10 ** 9), ((1 << 24) + 5, 1000), (22369622 + 77, 2500)])
def test_every_hit_once(n, every):
    import torch
    import pst_amd as P
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    hit = (i % every) == every // 2
    rec = torch.empty((n, 3), dtype=torch.int32, device="cuda")
    rec[:, 0] = torch.where(hit, 10, 21).int()
    rec[:, 1] = 30
    rec[:, 2] = i
    want = i[hit].cpu().numpy()
    for cap in {len(want), len(want) // 2}:
        out = torch.full((max(cap, 1) + 8,), -1, dtype=torch.int32, device="cuda")
        found = torch.zeros(1, dtype=torch.int64, device="cuda")
        P.ips_into(rec.view(-1).view(torch.uint8), n, 20, out, cap, found, "i32", "u32")
        torch.cuda.synchronize()
        assert int(found) == len(want)
        got = out.cpu().numpy()
        assert (got[cap:] == -1).all()
        if cap == len(want):
            assert np.array_equal(np.sort(got[:cap]), want)
        else:
            assert np.isin(got[:cap], want).all() and len(np.unique(got[:cap])) == cap
