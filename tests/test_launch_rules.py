"""Limits of the launch rules that no test system reaches, on the CPU: the header's own
functions, compiled for the host."""
import ctypes as C
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "device.h"
extern "C" int reaches(long long slots) { return hecmw33::flow_reaches(slots); }
"""


def test_fp32_sweeps_in_one_kernel_reach_their_records(tmp_path):
    """Offsets and the resource's size are 32-bit: 2 x 16 bytes per row slot, in slices of 16."""
    src, lib = str(tmp_path / "rules.hip"), str(tmp_path / "rules.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-x", "hip", "-std=c++17",
                    "-O1", "-fPIC", "-shared", "-I", os.path.join(ROOT, "frontistr_amd", "csrc"), src, "-o", lib],
                   check=True)
    L = C.CDLL(lib)
    L.reaches.argtypes = [C.c_longlong]
    most = 2 ** 32 // 32  # its size would be 0 in 32 bits
    assert L.reaches(16) and L.reaches(most - 16)
    assert not L.reaches(most) and not L.reaches(most + 16) and not L.reaches(2 ** 31 - 16)
