"""Batches that free slots and fill them again, in every launch form: within a
wave, across waves and across workgroups, over one round of a launch and
several, with as many workgroups as the device holds, fewer and more.  A
pointer that is published over the one still to be freed is never freed, and
one that a late clear wipes out neither: both leave pairs short of mallocs."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _stream(rng, n, order, nbatches=4):
    """A batch that fills n slots, then batches that free k = n / 2 of them and
    fill the same k again."""
    from gallatin_amd import BATCH_OP_DTYPE
    first = np.zeros(n, BATCH_OP_DTYPE)
    first["arg"], first["slot"] = 16, rng.permutation(n)
    ops, k = [first], n // 2
    for _ in range(nbatches):
        slots = rng.permutation(n)[:k]
        o = np.zeros(2 * k, BATCH_OP_DTYPE)
        if order == "pairs":  # free and fill side by side
            free_at = 2 * np.arange(k)
            fill_at = free_at + 1
        elif order == "reversed":  # the last slot freed is the first one filled
            free_at, fill_at = np.arange(k), 2 * k - 1 - np.arange(k)
        else:
            free_at, fill_at = np.sort(rng.permutation(2 * k).reshape(k, 2), axis=1).T
        o["kind"][free_at], o["slot"][free_at] = 1, slots
        o["slot"][fill_at] = slots
        o["arg"][fill_at] = 16 << rng.integers(0, 6, k)
        ops.append(o)
    off = np.concatenate([[0], np.cumsum([len(o) for o in ops])]).astype(np.uint64)
    return np.concatenate(ops), off


def _run(gpu, n, order, batched, threads, workgroups):
    import torch
    ops, off = _stream(np.random.default_rng(n), n, order)
    gpu.check_batch_stream(ops, off, n, persistent=False)
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(
        8 << 30, 3, print_info=False, flags=gpu.GAL_FLAG_NO_PAYLOAD_FENCE)
    st = gpu.BatchStream(ops, off, n)
    c = gpu.run_batches(a, st, threads=threads, batched=batched, workgroups=workgroups)
    torch.cuda.synchronize()
    c = c.cpu().tolist()
    assert c[gpu.CTR_MALLOCS] == c[gpu.CTR_PAIRS] == st.n_mallocs
    assert c[gpu.CTR_BAD] == c[gpu.CTR_MISSES] == c[gpu.CTR_TIMEOUTS] == 0
    assert int(st.ptrs.abs().sum()) == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()


@pytest.mark.parametrize("batched,threads", [(0, 256), (1, 256), (1, 1024), (2, 256), (2, 1024)])
@pytest.mark.parametrize("order", ["pairs", "reversed", "random"])
@pytest.mark.parametrize("n", [6, 200, 1024, 1026, 5001])
def test_a_batch_fills_what_it_frees(gpu, n, order, batched, threads):
    _run(gpu, n, order, batched, threads, 0)


@pytest.mark.parametrize("batched,threads", [(0, 256), (1, 512), (2, 512)])
@pytest.mark.parametrize("n,workgroups", [(5001, 1), (20_000, 3), (1_200_000, 4000)])
def test_with_a_given_number_of_workgroups(gpu, n, workgroups, batched, threads):
    _run(gpu, n, "random", batched, threads, workgroups)
