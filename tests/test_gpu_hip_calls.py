"""What the resident solves ask of HIP, and what they do when HIP refuses it."""
import pytest

from tests import hip_shim

pytestmark = pytest.mark.gpu


def test_kernel_attributes_do_not_depend_on_the_system(tmp_path):
    """A kernel's attributes belong to the process: two contexts on two threads would undo each
    other's between setting one and launching, so every solve sets the same."""
    out = hip_shim.run(tmp_path, """
for n in (2, 5, 9):
    for pc in (1, 3):
        m = fa.gen_hex8(n)
        m.set_precond(pc)
        m.set_iter(500)
        assert fa.hecmw_solve_krylov(m).error == 0
calls = val("attr_n").value
func = (ctypes.c_void_p * 256).in_dll(shim, "attr_func")
value = (ctypes.c_int * 256).in_dll(shim, "attr_value")
by = {}
for i in range(calls):
    by.setdefault(func[i], set()).add(value[i])
print("calls", calls, "most", max(len(v) for v in by.values()))
""")
    words = out[-1].split()
    assert int(words[1]) >= 6 and int(words[3]) == 1, out


SOLVE = """
def system():
    m = {make}
    m.set_precond({precond})
    m.set_method({method})
    m.set_iter(3000)
    m.set_resid(1e-10)
    m.X[:] = np.random.default_rng(5).standard_normal(m.X.size) * 1e-3
    return m
def solve(m):
    before = val("coop_calls").value
    r = fa.hecmw_solve_krylov(m)
    n = val("coop_calls").value - before
    print("iter", r.iter, "error", r.error, "coop", n)
    return r, n
m = system()
xr, info = restate.solve_krylov(m, x0=m.X.copy())
r, n = solve(m)
assert n > 0 and r.error == 0
val("coop_refuse").value = 1
a = system()
ra, n = solve(a)
assert n == 1 and ra.error == 0, "a refused launch"
assert abs(ra.iter - info["iter"]) <= 2 + 0.1 * info["iter"] * ({method} == 2) and ra.resid <= 1e-10
assert np.linalg.norm(a.X - xr) <= 1e-6 * np.linalg.norm(xr)
b = system()
rb, n = solve(b)
assert n > 0 and rb.error == 0 and np.array_equal(b.X, m.X), "the next solve is resident again"
val("gave_up").value = 1
c = system()
rc, n = solve(c)
assert n > 0 and rc.error == 0, "a wait that ran out"
assert rc.iter == ra.iter and rc.resid == ra.resid and np.array_equal(c.X, a.X)
d = system()
rd, n = solve(d)
assert n == 0 and rd.error == 0 and np.array_equal(d.X, a.X), "launches from then on"
print("done")
"""


@pytest.mark.parametrize("method,precond,make", [
    (1, 1, "fa.gen_hex8(5, kind='lognormal', seed=2)"), (1, 1, "fa.gen_hex8(12, kind='lognormal', seed=2)"),
    (2, 1, "fa.gen_hex8(9, kind='lognormal', seed=2)"), (1, 3, "fa.gen_hex8(9, kind='lognormal', seed=2)")])
def test_a_refused_launch_or_an_ended_wait_leaves_the_solve_to_the_launches(tmp_path, method, precond, make):
    """The same call succeeded before there were resident kernels, and does where HIP refuses a
    cooperative launch or a workgroup waits too long for the others: the launch-per-kernel solve
    starts again from x0 (the second time bit for bit what it was the first time)."""
    out = hip_shim.run(tmp_path, SOLVE.format(method=method, precond=precond, make=make))
    assert out[-1] == "done", out
