"""Build recipe of tests/payload/libpayload_kernels.so: the churn kernels' fill
and verify behind one test kernel.

    python -m tests.payload.build
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIB = os.path.join(HERE, "libpayload_kernels.so")


def build(verbose=False):
    sys.path.insert(0, ROOT)
    from gallatin_amd import build as hip_build
    tmp = LIB + ".tmp"
    cmd = [hip_build._hipcc(), *hip_build.HIP_FLAGS, "-shared",
           "-I", hip_build.INCLUDE, "-I", os.path.join(hip_build.HERE, "csrc"),
           os.path.join(HERE, "payload_kernels.hip"), "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
