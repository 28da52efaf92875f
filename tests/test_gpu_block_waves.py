"""Whole-block requests of many waves on the segments of one class, with more
lanes wanting blocks than a segment has left, in workgroups of one wave to
sixteen: blocks never overlap, no request misses, and every block comes back."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("partitions", [1, 8])
@pytest.mark.parametrize("threads", [64, 256, 1024])
@pytest.mark.parametrize("block,n", [(64 << 10, 1025), (64 << 10, 16_384), (2 * MIB, 1000)])
def test_many_waves_on_one_class(gpu, block, n, threads, partitions):
    import torch
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(16 << 30, 5, print_info=False,
                                                            partitions=partitions)
    sz = torch.full((n,), block, dtype=torch.int64, device="cuda")
    for _ in range(3):  # fresh segments, then ones whose blocks came back
        ptrs = a.malloc_bulk(sz, block_threads=threads)
        p = np.sort(ptrs.cpu().numpy().view(np.uint64))
        off = p - np.uint64(a.pool_base)
        assert (p != 0).all() and (off % np.uint64(block) == 0).all()
        assert (np.diff(off) >= block).all() and off[-1] + block <= a.num_segments * 16 * MIB
        a.free_bulk(ptrs, block_threads=threads)
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
