"""What a system that keeps the launches asks of the host: nothing of the resident solves."""
import pytest

from tests import hip_shim

pytestmark = pytest.mark.gpu

DIAG = """
import torch
m = fa.gen_hex8({n})
m.set_precond(3)
m.set_iter(3)
ctx = fa.DeviceContext()
ctx.load(m)
ia = m.Iarray.copy()
ia[m.I_FLAG_NUMFACT - 1] = ia[m.I_FLAG_SYMBFACT - 1] = 0
b = torch.from_numpy(m.B).cuda()
x = torch.zeros_like(b)
torch.cuda.synchronize()
before = val("malloc_calls").value
r = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
assert (r.iter, r.error) == (4, 3001)
print(m.N, ctx.info()["resident"], val("malloc_calls").value - before)
ctx.close()
"""


@pytest.mark.parametrize("n,resident,calls", [(55, 0, 1), (54, 256, 6)])
def test_diag_tasks_are_made_only_where_they_can_fit(tmp_path, n, resident, calls):
    """160 KB of LDS per workgroup hold 42 tasks of at most 16 rows: 172,032 nodes with 256
    workgroups.  Above that (56^3 = 175,616 nodes) a solve allocates the residual history only;
    below (55^3 = 166,375, whose tasks are full) it is resident, with three lists of tasks, the
    ring of z and the words of the exchange."""
    out = hip_shim.run(tmp_path, DIAG.format(n=n))[-1].split()
    assert (int(out[1]), int(out[2])) == (resident, calls), out
