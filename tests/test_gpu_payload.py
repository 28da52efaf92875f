"""The churn kernels' wave-wide fill and verify against host memory images: every
word of every lane's buffer is written once with its own pattern and nothing
beside it, and the verify counts exactly the words that differ."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "payload", "libpayload_kernels.so")
FULL = [512] * 64


def _cases():
    rng = np.random.default_rng(3)
    churn = np.maximum(1, np.floor(4096 ** rng.random(64))).astype(int)
    yield "one word", [0] * 37 + [1] + [0] * 26
    yield "largest", FULL
    yield "none", [0] * 64
    yield "last lane only", [0] * 63 + [511]
    yield "all one word", [1] * 64
    yield "all two words", [2] * 64
    yield "odd and even", [1 + l % 9 for l in range(64)]
    yield "one ends on a word of the map", [128, 1] + [127] * 62
    yield "churn sizes", ((churn + 7) // 8).tolist()
    yield "churn sizes, half", np.where(rng.random(64) < 0.5, (churn + 7) // 8, 0).tolist()


@pytest.mark.parametrize("name,words", list(_cases()), ids=[c[0] for c in _cases()])
def test_fill_and_verify_touch_exactly_the_buffers(gpu, name, words):
    import torch
    if not os.path.exists(LIB):
        pytest.fail("tests/payload/libpayload_kernels.so is not built (run build())")
    lib = ctypes.CDLL(LIB)
    lib.payload_run.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int]
    rng = np.random.default_rng(5)
    # buffers in random order with a 16-byte gap after each
    start, at = np.zeros(64, np.int64), 2
    for l in rng.permutation(64):
        start[l] = at
        at += (words[l] + 1) // 2 * 2 + 2
    image = np.full(at + 2, -1, np.int64)
    mem = torch.from_numpy(image).cuda()
    pats = rng.integers(1, 1 << 62, 64)
    ptrs = torch.from_numpy(mem.data_ptr() + 8 * start).cuda()
    w = torch.from_numpy(np.asarray(words, np.int32)).cuda()
    p = torch.from_numpy(pats).cuda()
    bad = torch.zeros(64, dtype=torch.int32, device="cuda")

    def run(verify):
        assert lib.payload_run(ptrs.data_ptr(), w.data_ptr(), p.data_ptr(), bad.data_ptr(),
                               verify) == 0
        return int(bad.sum())

    run(0)
    # the upper half of an odd buffer's last 16 bytes belongs to the buffer
    for l in range(64):
        image[start[l]:start[l] + (words[l] + 1) // 2 * 2] = pats[l]
    assert np.array_equal(mem.cpu().numpy(), image)
    assert run(1) == 0
    # some words changed: the verify counts them, and no word past a buffer
    owned = np.concatenate([np.arange(start[l], start[l] + words[l]) for l in range(64)])
    wrong = image.copy()
    other = np.ones(len(image), bool)
    other[owned] = False
    wrong[other] += 1
    hit = rng.permutation(owned)[:len(owned) // 7 + (len(owned) > 0)]
    wrong[hit] ^= 1 << 40
    mem.copy_(torch.from_numpy(wrong))
    assert run(1) == len(hit)
