"""A program's own calls of the chaining table's device functions, in the forms
it always had: chaining_block::init(defaultKey) and attach_block(link)."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "chain_calls",
                   "libchain_kernels.so")


def test_init_and_attach_block():
    import torch
    torch.cuda.set_device(0)
    if not os.path.exists(LIB):
        pytest.fail("tests/chain_calls/libchain_kernels.so is not built (run build())")
    errors = (ctypes.c_ulonglong * 8)()
    assert ctypes.CDLL(LIB).chain_calls(errors) == 0
    assert list(errors) == [0] * 8
