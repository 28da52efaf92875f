"""The waits that put a batch's stores in order (CPU; reads the source).

`s_waitcnt` is no barrier to the compiler: a relaxed store or LDS addition may
be moved across it.  Where the order matters to another wave, a signal fence
(or the workgroup barrier) stands on each side."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_wait_of_the_batch_kernels_is_fenced():
    with open(os.path.join(ROOT, "gallatin_amd", "csrc", "batches.hip")) as f:
        lines = [re.sub(r"//.*", "", l).strip() for l in f]
    lines = [l for l in lines if l]
    waits = [i for i, l in enumerate(lines) if l.startswith("__builtin_amdgcn_s_waitcnt(0)")]
    assert len(waits) >= 5
    fence = "__atomic_signal_fence(__ATOMIC_SEQ_CST);"
    for i in waits:
        assert lines[i - 1] == fence, lines[i - 1:i + 2]
        assert lines[i + 1] in (fence, "__syncthreads();"), lines[i - 1:i + 2]
