"""Counters summed per workgroup: the counts of launches whose last workgroup
or wave is partly empty, at the edges of waves and workgroups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 1000])
def test_serving_step_counts_every_operation(gpu, n):
    import torch
    from gallatin_amd import serving as SV
    gpu.init_global_allocator(16 << 30, 9, print_info=False)
    try:
        sv = SV.Serving(512, seed=4)
        c = torch.zeros(16, dtype=torch.int64, device="cuda")
        sv.step(0, n, 0, 0.0, n, c)
        sv.step(1, 0, 0, 1.0, 0, c)  # 2^32 wraps to 0: no session ends
        torch.cuda.synchronize()
        c = c.tolist()
        held = sv.check()
        assert c[0] == min(n, 512) and c[0] + c[1] == n and c[2] == 0
        assert held["live"] == c[0] and held["words"] == c[3] and held["bad"] == 0
        assert c[4] == 0 and c[6] == 0 and c[7] == 0 and c[5] >= c[0]
        assert c[8] + c[9] + c[10] == n and c[11] == 0
        sv.destroy()
    finally:
        gpu.free_global_allocator()


@pytest.mark.parametrize("threads,batched", [(256, 0), (256, 1), (512, 1), (1024, 1), (256, 2)])
@pytest.mark.parametrize("n", [1, 65, 1023, 1025, 5000])
def test_stream_counts_every_request(gpu, n, threads, batched):
    import torch
    from gallatin_amd import BATCH_OP_DTYPE
    ops = np.zeros(n + n // 2, BATCH_OP_DTYPE)
    ops["arg"][:n] = 16
    ops["slot"][:n] = np.arange(n)
    ops["kind"][n:] = 1
    ops["slot"][n:] = np.arange(n // 2)
    a = gpu.Gallatin(16 << 20, 16, 4096).generate_on_device(8 << 30, 3, print_info=False)
    st = gpu.BatchStream(ops, [0, n, len(ops)], n)
    c = torch.zeros(gpu.CTR_COUNT, dtype=torch.int64, device="cuda")
    plan = gpu.BatchPlan(a, st, c, threads=threads, batched=batched)
    for k in range(1, 4):
        plan.launch()
        torch.cuda.synchronize()
        v = c.tolist()
        assert v[:5] == [k * n, 0, 0, 16 * k * n, k * n]  # half freed by ops, half by the cleanup
        assert v[5] == 0 and v[6] == 0
    plan.destroy()
    a.free_on_device()
