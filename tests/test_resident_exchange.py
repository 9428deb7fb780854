"""The rules by which the resident kernels exchange vectors (csrc/resident.h), on the CPU: the
header's own functions, compiled for the host, against models of the memory around them."""
import ctypes as C
import itertools
import os
import struct
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "resident.h"
using namespace hecmw33;
extern "C" int missing1(const double* x) {
  return missing<1>(*reinterpret_cast<const double(*)[3]>(x), true);
}
extern "C" int missing2(const double* x, int with_z) {
  return missing<2>(*reinterpret_cast<const double(*)[6]>(x), with_z != 0);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = str(d / "rules.hip"), str(d / "rules.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-x", "hip", "-std=c++17",
                    "-O1", "-fPIC", "-shared", "-I", os.path.join(ROOT, "frontistr_amd", "csrc"), src, "-o", lib],
                   check=True)
    L = C.CDLL(lib)
    L.missing1.argtypes = [C.c_void_p]
    L.missing2.argtypes = [C.c_void_p, C.c_int]
    return L


MARK = struct.unpack("<d", struct.pack("<Q", 0x7FFADEAD << 32))[0]


def _is_mark(a):
    return a.view(np.uint64) >> np.uint64(32) == 0x7FFADEAD


@pytest.mark.parametrize("with_z", [True, False])
def test_a_record_from_lines_of_different_age_is_asked_for_again(rules, with_z):
    """A record {z0 z1 z2 w0 w1 w2} comes in three loads of two entries.  Each may be served by
    a line of any age: of the backward sweep (any of z marked, w marked), of this sweep
    (z there, any of w marked) or of memory now.  No mark that the sweep uses gets through, and
    a record without one is not asked for again."""
    now = np.array([1.0, 2.0, 3.0, 4.0, 5.0, 6.0])
    ages = []
    for z in itertools.product([False, True], repeat=3):  # True: marked
        ages.append(np.array(list(z) + [True] * 3))
    for w in itertools.product([False, True], repeat=3):
        ages.append(np.array([False] * 3 + list(w)))
    for pick in itertools.product(range(len(ages)), repeat=3):
        x = now.copy()
        for load, age in enumerate(pick):
            s = slice(2 * load, 2 * load + 2)
            x[s] = np.where(ages[age][s], MARK, now[s])
        used = _is_mark(x) if with_z else _is_mark(x)[3:]
        assert bool(rules.missing2(x.ctypes.data, int(with_z))) == bool(used.any()), x
        assert bool(rules.missing1(x.ctypes.data)) == bool(_is_mark(x[:3]).any())


def test_values_that_are_not_marks_are_taken(rules):
    x = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 5e-324])
    assert not rules.missing2(x.ctypes.data, 1) and not rules.missing1(x.ctypes.data)
