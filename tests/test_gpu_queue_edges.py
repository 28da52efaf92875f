"""Queue and ring of queues at the sizes where a wave's group of nodes ends:
one item, whole waves, one item past them; more dequeues than items, and
several passes, so that every dummy node is left and freed by two groups."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ring,smallest", [(False, 16), (True, 16), (False, 128)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 4097])
def test_every_item_once_and_no_node_lost(gpu, n, ring, smallest):
    import torch
    a = gpu.Gallatin(16 << 20, smallest, 4096).generate_on_device(4 << 30, 21, print_info=False)
    q = gpu.Queue(a, ring=ring)
    for k in range(3):
        items = torch.arange(1, n + 1, dtype=torch.int64, device="cuda") + 1000000 * k
        ok = q.enqueue(items)
        taken = []
        # a ring's dequeue looks at one queue only: a few calls reach them all
        for _ in range(16 if ring else 1):
            out, got = q.dequeue(n + 70)
            torch.cuda.synchronize()
            taken.append(out[got.bool()].cpu().numpy())
            if sum(map(len, taken)) == n:
                break
        assert bool(ok.all())
        assert np.array_equal(np.sort(np.concatenate(taken)), items.cpu().numpy())
        # half stays in the queue for the next pass's first dequeues to leave
        q.enqueue(items[: n // 2])
        out, got = q.dequeue(4 * n + 64)
        torch.cuda.synchronize()
        assert ring or int(got.sum()) == n // 2
        while ring and int(got.sum()):
            out, got = q.dequeue(4 * n + 64)
            torch.cuda.synchronize()
    q.destroy()
    a.drain()
    H.check_fresh(a)
    a.free_on_device()


def test_items_left_in_the_queue_are_freed(gpu):
    import torch
    a = gpu.Gallatin(16 << 20, 16, 4096).generate_on_device(4 << 30, 21, print_info=False)
    q = gpu.Queue(a)
    q.enqueue(torch.arange(1, 1001, dtype=torch.int64, device="cuda"))
    out, got = q.dequeue(130)
    torch.cuda.synchronize()
    assert bool(got.all()) and len(set(out.cpu().tolist())) == 130
    q.destroy()
    a.drain()
    H.check_fresh(a)
    a.free_on_device()
