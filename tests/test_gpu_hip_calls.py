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
