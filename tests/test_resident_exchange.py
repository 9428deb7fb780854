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
extern "C" int drops(int copy) { return drops_lines(copy); }
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


class Ring:
    """One record of each of four copies, and what the caches may hold of it at worst: every
    state that a load since the lines were last dropped can have seen, whatever the load's
    scope.  The sweeps' accesses in their order (k_resident_cg, k_resident_bicg)."""

    def __init__(self, rules, par):
        self.rules, self.par, self.n = rules, par, 0
        self.mem = [("mark", "mark")] * 4
        self.lines = [set() for _ in range(4)]

    def drop(self):
        self.lines = [set() for _ in range(4)]

    def enter(self, cp):
        if self.rules.drops(cp):
            self.drop()

    def next(self):
        return (self.par + 1) % 4

    def load(self, cp):
        self.lines[cp].add(self.mem[cp])

    def put(self, cp, z=None, w=None):
        z0, w0 = self.mem[cp]
        self.mem[cp] = (z or z0, w or w0)

    def look(self, cp, now, field):
        """A gather through the caches: nothing but a mark or the present value."""
        seen = {s[field] for s in self.lines[cp] | {self.mem[cp]}}
        assert seen <= {"mark", now}, (cp, seen, now)

    def backward(self, after_refresh=False, reads_last=False):
        last, self.par = self.par, self.next()
        self.enter(self.par)
        self.n += 1
        z = "z%d" % self.n
        for _ in range(2):  # before and after the record is written
            self.load(self.par)
            self.look(self.par, z, 0)
            if reads_last:  # another row of the line may have been marked or not
                self.load(last)
            self.put(self.par, z=z)
        self.put(last, z="mark", w="mark")
        if after_refresh:
            self.put(self.par, w="mark")
            self.drop()

    def forward(self):
        w = "w%d" % self.n
        for _ in range(2):
            self.load(self.par)
            self.look(self.par, "z%d" % self.n, 0)
            self.look(self.par, w, 1)
            self.put(self.par, w=w)

    def refresh(self):
        cp = self.next()
        self.enter(cp)
        self.n += 1
        u = "u%d" % self.n
        for _ in range(2):
            self.load(cp)
            self.look(cp, u, 1)
            self.put(cp, w=u)


@pytest.mark.parametrize("par", [0, 1, 2, 3])
@pytest.mark.parametrize("period", [3, 4, 5, 1000])
def test_cg_looks_find_no_old_value_in_the_caches(rules, par, period):
    r = Ring(rules, par)
    fresh = True
    for it in range(40):
        if fresh:
            r.refresh()
        r.backward(after_refresh=fresh)
        r.forward()
        fresh = it % period == period - 1


@pytest.mark.parametrize("par", [0, 2])  # as the solve starts, and as its launches end
@pytest.mark.parametrize("period", [1, 2, 3, 1000])
def test_bicgstab_looks_find_no_old_value_in_the_caches(rules, par, period):
    r = Ring(rules, par)
    fresh = True
    for it in range(40):
        if fresh:
            r.refresh()
        r.backward(after_refresh=fresh)
        r.forward()
        r.backward(reads_last=True)
        r.forward()
        r.load(r.par)  # x += omega s^
        fresh = it % period == period - 1
