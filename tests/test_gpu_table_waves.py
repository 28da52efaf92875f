"""Hash table operations where a wave's lanes read buckets together: whole and
partial waves, few and many keys per bucket, splits under way, keys that are
absent, against a dict."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def glob(gpu):
    gpu.init_global_allocator(8 << 30, 42, print_info=False)
    yield gpu
    gpu.free_global_allocator()


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("n", [1, 7, 8, 63, 64, 65, 255, 1000, 40007])
def test_rounds_of_updates_match_a_dict(glob, n, kind):
    import torch
    rng = np.random.default_rng(n)
    t = glob.Table(kind=kind, seed=9)
    want = {}
    cuda = lambda a: torch.from_numpy(a.astype(np.int64)).cuda()  # noqa: E731
    for rnd in range(4):
        keys = rng.choice(np.arange(1, 6 * n + 1), n, replace=False)
        vals = rng.integers(1, 1 << 62, n)
        ok = t.insert(cuda(keys), cuda(vals))
        assert bool(ok.all())
        want.update(zip(keys.tolist(), vals.tolist()))
        gone = rng.choice(np.arange(1, 6 * n + 1), n, replace=False)
        ok = t.remove(cuda(gone)).cpu().numpy()
        assert np.array_equal(ok, [int(k in want) for k in gone.tolist()])
        for k in gone.tolist():
            want.pop(k, None)
        asked = rng.permutation(np.arange(1, 6 * n + 1))
        got, found = (x.cpu().numpy() for x in t.query(cuda(asked)))
        assert np.array_equal(found, [int(k in want) for k in asked.tolist()])
        assert np.array_equal(got, [want.get(k, 0) for k in asked.tolist()])
    s = t.stats()
    assert s["keys"] == len(want) and s["failed"] == 0
    t.destroy()


def test_many_lanes_on_one_key(glob):
    import torch
    t = glob.Table(kind=0, seed=9)
    keys = torch.full((300,), 77, dtype=torch.int64, device="cuda")
    vals = torch.arange(1, 301, dtype=torch.int64, device="cuda")
    assert bool(t.insert(keys, vals).all())
    got, found = t.query(keys[:5])
    assert bool(found.all()) and len(set(got.tolist())) == 1 and 1 <= int(got[0]) <= 300
    assert int(t.remove(keys).sum()) == 1
    assert t.stats()["keys"] == 0
    t.destroy()
