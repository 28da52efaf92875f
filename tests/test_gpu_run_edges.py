"""Runs of per-thread batches whose mallocs and frees fill waves whole or in
part, up to the largest batch of a run and just past it."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("batches", [
    [(640, 0), (0, 640), (640, 0), (639, 1), (1, 639), (0, 640)],
    [(320, 0), (320, 320), (321, 319), (319, 321), (64, 64), (65, 63), (63, 65)],
    [(640, 0), (641, 0), (0, 641), (0, 640), (5, 0), (0, 5), (1, 0), (0, 1)],
    [(577, 0), (63, 577), (577, 63), (0, 577)],
], ids=["whole", "halves", "past the largest", "one wave more"])
def test_mallocs_and_frees_side_by_side(gpu, batches):
    import torch
    rng = np.random.default_rng(7)
    live, slots, ops, off = [], 0, [], [0]
    for mallocs, frees in batches:
        o = np.zeros(mallocs + frees, gpu.BATCH_OP_DTYPE)
        at = rng.permutation(len(o))
        live = list(rng.permutation(live))
        o["kind"][at[:frees]] = 1
        o["slot"][at[:frees]] = live[:frees]
        assert len(live) >= frees
        o["slot"][at[frees:]] = slots + np.arange(mallocs)
        o["arg"][at[frees:]] = 16 << rng.integers(0, 9, mallocs)
        live = live[frees:] + list(range(slots, slots + mallocs))
        slots += mallocs
        ops.append(o)
        off.append(off[-1] + len(o))
    st = gpu.BatchStream(np.concatenate(ops), off, slots)
    a = gpu.Gallatin(16 * MIB, 16, 4096).generate_on_device(
        8 << 30, 3, print_info=False, flags=gpu.GAL_FLAG_NO_PAYLOAD_FENCE)
    for _ in range(3):
        c = gpu.run_batches(a, st, batched=0)
        torch.cuda.synchronize()
        c = c.cpu().tolist()
        assert c[gpu.CTR_MALLOCS] == c[gpu.CTR_PAIRS] == slots
        assert c[gpu.CTR_BAD] == c[gpu.CTR_MISSES] == c[gpu.CTR_TIMEOUTS] == 0
        assert int(st.ptrs.abs().sum()) == 0
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
