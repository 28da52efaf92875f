"""No kernel of the library or of the test programs shifts a 64-bit value by its
last vector register (CPU; compiles every source to assembly)."""
import glob
import os
from concurrent.futures import ThreadPoolExecutor

import pytest

from gallatin_amd import build as B

SOURCES = sorted(glob.glob(os.path.join(B.HERE, "csrc", "*.hip")) +
                 glob.glob(os.path.join(B.ROOT, "tests", "*", "*.hip")))

KERNEL = """\
leaf:                                   ; @leaf
\tv_lshlrev_b64 v[2:3], v{leaf}, -1
.Lfunc_end0:
k:                                      ; @k
\tv_lshrrev_b64 v[2:3], v{own}, v[4:5]
\tv_lshlrev_b32_e32 v1, v{top}, v1
\ts_add_u32 s0, s0, leaf@rel32@lo+4
.Lfunc_end1:
\t.amdhsa_kernel k
\t\t.amdhsa_next_free_vgpr {used}
\t.end_amdhsa_kernel
"""


@pytest.mark.parametrize("used,own,leaf,bad", [
    (120, 119, 0, ["k"]), (120, 0, 119, ["leaf"]), (113, 119, 119, ["k", "leaf"]),
    (120, 118, 111, []), (121, 119, 119, []), (128, 119, 119, []), (8, 7, 6, ["k"]),
])
def test_finds_the_form_in_a_kernel_and_what_it_calls(used, own, leaf, bad):
    last = (used + 7) // 8 * 8 - 1
    text = KERNEL.format(used=used, own=own, leaf=leaf, top=last)
    assert B.shift_hazards(text) == [("k", f, last) for f in bad]


def test_no_kernel_shifts_by_its_last_register(tmp_path):
    def one(src):
        return B.shift_hazards(B.assembly(src, str(tmp_path / (os.path.basename(src) + ".s"))))

    with ThreadPoolExecutor(4) as pool:
        found = dict(zip(SOURCES, pool.map(one, SOURCES)))
    assert {os.path.basename(s): f for s, f in found.items() if f} == {}
