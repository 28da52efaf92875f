"""Chains whose blocks are attached with a pair in them: many inserts at once
into one, a few and many chains, for every key width and block size, with and
without preallocated first blocks.  A chain of c keys has ceil(c / size)
blocks, every pair is found, and the allocator drains to fresh."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def glob(gpu):
    gpu.init_global_allocator(8 << 30, 42, print_info=False)
    yield gpu
    g = gpu.global_allocator()
    g.drain()
    H.check_fresh(g)
    gpu.free_global_allocator()


@pytest.mark.parametrize("prealloc", [False, True])
@pytest.mark.parametrize("chains", [1, 7, 5000])
@pytest.mark.parametrize("n", [1, 4, 65, 3000])
@pytest.mark.parametrize("kind", [0, 1, 2, 3, 4])
def test_concurrent_inserts(glob, kind, n, chains, prealloc):
    import torch
    width, size = glob.ChainTable.KINDS[kind]
    dt = np.int64 if width == 8 else np.int32
    keys = np.random.default_rng(n).permutation(n).astype(dt) + 1
    t = glob.ChainTable(kind, nslots=chains * size, seed=3, prealloc=prealloc)
    k, v = torch.from_numpy(keys).cuda(), torch.from_numpy(keys * 3).cuda()
    assert bool(t.insert(k, v).all())
    got, found = t.query(k)
    assert bool(found.all()) and torch.equal(got, v)
    _, found = t.query(k + n)
    assert not bool(found.any())
    blocks = t.lengths().cpu().numpy()
    s = t.stats()
    assert s["failed"] == 0 and s["blocks"] == blocks.sum()
    if chains == 1:
        assert blocks[0] == -(-n // size)
    # no chain has room for a whole block more than its keys need
    assert blocks.sum() <= (n + chains * (size - 1)) / size + (chains if prealloc else 0)
    t.destroy()
