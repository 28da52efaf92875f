"""Session slots per wave: tables of sessions around the sizes at which a wave
takes more slots, and smaller than one wave's share.  Every word of every live
session reads back and nothing is left allocated."""
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sessions", [1, 7, 9, 2049, 131071, 131073, 262145, 524289])
def test_sessions_per_wave(gpu, sessions):
    import torch
    from gallatin_amd import serving as SV
    gpu.init_global_allocator(16 << 30, 9, print_info=False)
    try:
        r = SV.run(torch, steps=12, warmup=4, seed=3, max_sessions=sessions,
                   arrivals_mean=max(1, min(sessions // 4, 4000)), p_end=0.1, ht_ops=512,
                   reserve_fraction=0.0)
        c = r["counters"]
        assert r["session_words_bad"] == 0 and r["live_sessions"] == c["admitted"] - c["ended"]
        assert c["words"] > 0 and c["chunk_failed"] == 0 and c["words_refused"] == 0
        assert c["ht_inserted"] + c["ht_removed"] + c["ht_absent"] + c["ht_failed"] == 16 * 512
        g = gpu.global_allocator()
        g.drain()
        H.check_fresh(g)
    finally:
        gpu.free_global_allocator()
