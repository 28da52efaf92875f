"""A wave's whole-block and multi-segment frees run side by side: every run and
every completed block comes back exactly once, whatever else the wave frees."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("partitions", [1, 8])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
def test_mixed_wave_frees_bring_everything_back(gpu, n, partitions):
    import torch
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(32 << 30, 5, print_info=False,
                                                            partitions=partitions)
    rng = np.random.default_rng(n)
    # runs of 2 to 5 segments, whole blocks of every class, runs of largest
    # slices, single slices and (as nullptr) nothing
    sizes = np.array([20 * MIB, 16, 64 << 10, 70 * MIB, 16 * MIB, 4096, 3 * MIB, 100 << 10,
                      33 * MIB, 1 * MIB, 12000, 50 * MIB])
    pick = np.resize(sizes, n)
    for k in range(3):
        before = a.stats()
        sz = torch.from_numpy(rng.permutation(pick).astype(np.int64)).cuda()
        p = a.malloc_bulk(sz)
        torch.cuda.synchronize()
        ptrs = p.cpu().numpy()
        assert (ptrs != 0).all() and len(set(ptrs.tolist())) == n
        keep = rng.random(n) < 0.1
        order = rng.permutation(n)
        first = np.where(keep, 0, ptrs)[order]
        a.free_bulk(torch.from_numpy(first).cuda())
        a.free_bulk(torch.from_numpy(np.where(keep, ptrs, 0)).cuda())
        torch.cuda.synchronize()
        after = a.stats()
        assert after["errors"] == before["errors"] == 0
        runs = (sz.cpu().numpy() + 16 * MIB - 1) // (16 * MIB)
        assert after["segments_released"] - before["segments_released"] >= runs[runs > 1].sum()
        assert a.info()["segments_multi"] == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
