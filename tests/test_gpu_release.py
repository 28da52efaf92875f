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
