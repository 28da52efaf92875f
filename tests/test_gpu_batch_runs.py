"""Consecutive small batches served by one launch: run lengths and batch sizes
at their limits, empty batches, slots used again in later batches, and a pool
so small that a batch's mallocs need the memory its frees give back."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _stream(rng, counts, max_live, sizes):
    """Batches of the given op counts over a table of max_live slots, each slot
    used again as soon as a batch after its free comes."""
    from gallatin_amd import BATCH_OP_DTYPE
    free_slots, live = list(range(max_live)), []
    ops, offsets = [], [0]
    for n in counts:
        o = np.zeros(n, BATCH_OP_DTYPE)
        gone, new = [], []
        for i in range(n):
            if live and (not free_slots or rng.random() < 0.5):
                s = live.pop(rng.integers(len(live)))
                o[i] = (0, 1, s)
                gone.append(s)
            elif free_slots:
                s = free_slots.pop(rng.integers(len(free_slots)))
                o[i] = (sizes[rng.integers(len(sizes))], 0, s)
                new.append(s)
            else:
                o = o[:i]
                break
        live += new
        free_slots += gone
        ops.append(o)
        offsets.append(offsets[-1] + len(o))
    return np.concatenate(ops), np.array(offsets, np.uint64), max_live


@pytest.mark.parametrize("batched,threads", [(0, 256), (1, 256), (1, 512), (1, 1024), (2, 256)])
@pytest.mark.parametrize("name,counts", [
    ("one small", [5]),
    ("limits", [1, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1]),
    ("empty ones", [0, 3, 0, 0, 64, 0, 65, 0]),
    ("all frees of two passes", [1024, 1024, 1024, 1024]),
    ("longer than a run", [3] * 300),
    ("run, large, run", [7] * 130 + [3000] + [9] * 128),
], ids=lambda x: x if isinstance(x, str) else "")
def test_runs_of_batches(gpu, name, counts, batched, threads):
    import torch
    rng = np.random.default_rng(len(counts))
    ops, off, nslots = _stream(rng, counts, 1500, [16, 100, 4096, 5000, 70000, 20 * MIB])
    gpu.check_batch_stream(ops, off, nslots, persistent=False)
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(
        24 << 30, 3, print_info=False, slots_min=32, flags=gpu.GAL_FLAG_NO_PAYLOAD_FENCE)
    st = gpu.BatchStream(ops, off, nslots)
    for _ in range(3):
        c = gpu.run_batches(a, st, threads=threads, batched=batched)
        torch.cuda.synchronize()
        c = c.cpu().tolist()
        assert c[gpu.CTR_MALLOCS] == c[gpu.CTR_PAIRS] == st.n_mallocs
        assert c[gpu.CTR_BAD] == c[gpu.CTR_MISSES] == c[gpu.CTR_TIMEOUTS] == 0
        assert int(st.ptrs.abs().sum()) == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()


def test_a_batch_allocates_what_it_frees(gpu):
    import torch
    from gallatin_amd import BATCH_OP_DTYPE
    # Twenty batches that each free the whole free pool and take it again.
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(
        2 << 30, 3, print_info=False, flags=gpu.GAL_FLAG_NO_PAYLOAD_FENCE)
    room = a.info()["segments_free"]
    ops = [np.array([(16 * MIB * room, 0, 0)], BATCH_OP_DTYPE)]
    for b in range(1, 21):
        ops.append(np.array([(0, 1, b - 1), (16 * MIB * room, 0, b)], BATCH_OP_DTYPE))
    off = np.concatenate([[0], np.cumsum([len(o) for o in ops])]).astype(np.uint64)
    st = gpu.BatchStream(np.concatenate(ops), off, 21)
    c = gpu.run_batches(a, st, threads=256, batched=0)
    torch.cuda.synchronize()
    c = c.cpu().tolist()
    assert c[gpu.CTR_MISSES] == 0 and c[gpu.CTR_PAIRS] == 21 and c[gpu.CTR_BAD] == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
