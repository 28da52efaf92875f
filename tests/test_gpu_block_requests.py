"""Whole-block requests of a wave served together: every class from many blocks
per segment to one, with fewer, as many and more lanes than a segment has
blocks, on fresh and on partly used segments.  Blocks never overlap, are
aligned to their size, and come back."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("partitions", [1, 8])
@pytest.mark.parametrize("n", [1, 3, 64, 65, 200])
@pytest.mark.parametrize("block", [64 << 10, 1 * MIB, 4 * MIB, 8 * MIB, 16 * MIB])
def test_blocks_of_one_class(gpu, block, n, partitions):
    import torch
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(16 << 30, 5, print_info=False,
                                                            partitions=partitions)
    sz = torch.full((n,), block - 7, dtype=torch.int64, device="cuda")
    held = []
    for k in range(3):
        ptrs = a.malloc_bulk(sz)
        torch.cuda.synchronize()
        held.append(ptrs)
        if k == 1:  # the next pass finds segments with some blocks free
            a.free_bulk(held.pop(0))
    p = np.sort(torch.cat(held).cpu().numpy().view(np.uint64))
    off = p - np.uint64(a.pool_base)
    assert (p != 0).all() and (off % np.uint64(block) == 0).all()
    assert (np.diff(off) >= block).all() and off[-1] + block <= a.num_segments * 16 * MIB
    for ptrs in held:
        a.free_bulk(ptrs)
    a.drain()
    H.check_fresh(a)
    a.free_on_device()


def test_pool_runs_out_and_recovers(gpu):
    import torch
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(8 << 30, 5, print_info=False)
    sz = torch.full((700,), 16 * MIB, dtype=torch.int64, device="cuda")
    for _ in range(3):
        p = a.malloc_bulk(sz)
        torch.cuda.synchronize()
        got = p[p != 0]
        assert 300 < got.numel() < 512 and len(set(got.cpu().tolist())) == got.numel()
        a.free_bulk(p)
    torch.cuda.synchronize()
    assert a.info()["errors"] == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
