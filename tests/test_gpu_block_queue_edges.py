"""Block queue: launches whose last node is exactly full, one short or one
past, and whose waves meet full nodes in different lanes, filled and emptied
several times without the nodes being given back in between."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,node", [(0, 256), (1, 16)])
@pytest.mark.parametrize("nodes,past", [(1, -1), (1, 0), (1, 1), (3, 0), (9, 5), (60, -7)])
def test_nodes_filled_to_their_edge(gpu, kind, node, nodes, past):
    import torch
    gpu.init_global_allocator(8 << 30, 5, print_info=False)
    try:
        q = gpu.BlockQueue(kind)
        n = nodes * node + past
        for k in range(3):
            items = torch.arange(1, n + 1, dtype=torch.int64, device="cuda") + k * n
            assert bool(q.enqueue(items).all())
            out, got = q.dequeue(n)
            assert bool(got.all())
            assert torch.equal(torch.sort(out)[0].cpu(), items.cpu())
            assert not bool(q.dequeue(1)[1].any())
        q.reclaim()
        q.destroy()
        g = gpu.global_allocator()
        g.drain()
        from tests import helpers as H
        H.check_fresh(g)
    finally:
        gpu.free_global_allocator()
