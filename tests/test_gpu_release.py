"""Payload survives frees whose L2 write-back is shared between the waves of
an XCD: launches around the size from which waves share it, on one partition
(every free needs it) and on one per XCD, per thread and in workgroup
batches.  Every allocation is filled and verified by the churn itself."""
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("partitions", [1, 8])
@pytest.mark.parametrize("n", [32704, 32768, 33001, 300007])
def test_churn_payload_around_the_sharing_threshold(gpu, n, partitions, batched):
    import torch
    a = gpu.Gallatin(16 << 20, 16, 4096).generate_on_device(8 << 30, 7, print_info=False,
                                                           partitions=partitions)
    for seed in (1, 2):
        run = a.run_churn_batched if batched else a.run_churn
        c = run(seed, n, 4)
        torch.cuda.synchronize()
        c = c.cpu().tolist()
        assert c[gpu.CTR_BAD] == 0 and c[gpu.CTR_MISSES] == 0
        assert c[gpu.CTR_PAIRS] == c[gpu.CTR_MALLOCS] >= n
    a.drain()
    H.check_fresh(a)
    a.free_on_device()


def test_pinned_blocks_come_back_from_a_slow_pool(gpu):
    """Waves of a launch that allocates and frees at once add to full blocks
    while they are replaced; a pool in host memory holds them up longest.
    Every block pinned meanwhile is accounted for afterwards."""
    import torch
    for k in range(12):
        a = gpu.Gallatin(16 << 20, 16, 4096).generate_on_device_host(4 << 30, 42,
                                                                    print_info=False)
        try:
            a.run_plain(1 << 18, 16)
            a.run_churn(5 + k, 1 << 16, 4)
            torch.cuda.synchronize()
            a.drain()
            H.check_fresh(a)
        finally:
            a.free_on_device()
