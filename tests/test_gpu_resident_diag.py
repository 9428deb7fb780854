"""The resident CG with block-diagonal scaling (csrc/resident_diag.hip) against the plain-C
restatement of hecmw_solve_CG (oracle/restate.c) and against the launch-per-kernel solve,
which a system with an external node takes.

The sums are formed in another order: rounding of about 1e-16 per operation, 1e3
operations deep and amplified by the condition of these systems (up to 1e5), hence
1e-8 on the first fifteen residuals above 1e-7; the residual of a CG with this scaling
oscillates, so the iteration that crosses the tolerance may shift by a few: 3 or 2% of
the count.  Solutions to a 1e-10 residual agree to 1e-6.
"""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate
from tests.systems import random_system
from tests.test_gpu_resident import _device_solve, _same_start, _with_external_node

pytestmark = pytest.mark.gpu

# name: system, workgroups, iterations at most.  Tasks of 16 rows on 4 waves per workgroup
SYSTEMS = {
    "one_element": (lambda: fa.gen_hex8(1), 1, 3000),                              # one task
    "ragged_rows": (lambda: fa.gen_tet10(3, 2, 4, seed=1)[0], None, 3000),         # N % 4 != 0, long rows
    "one_group": (lambda: fa.gen_hex8(4, kind="lognormal", seed=2), 1, 3000),      # two tasks of a wave
    "few_groups": (lambda: fa.gen_hex8(9, kind="lognormal", seed=2), None, 3000),
    "one_task": (lambda: fa.gen_hex8(19), None, 3000),                             # more than 64 workgroups
    "two_tasks": (lambda: fa.gen_hex8(27), 256, 3000),
    "three_tasks": (lambda: fa.gen_hex8(33), 256, 120),
    "read_again": (lambda: fa.gen_hex8(41), 256, 60),                              # more tasks than registers
    "wide_rows": (lambda: random_system(203, deg=100, seed=3), None, 3000),        # four rows on almost 64 lanes
    "odd_rows": (lambda: random_system(777, deg=9, seed=5), None, 3000),
}


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_resident_diag_cg_matches_the_restatement(name):
    make, groups, maxit = SYSTEMS[name]
    m = make()
    m.set_iter(maxit)
    m.set_precond(3)
    m.set_resid(1e-10)
    x0 = np.random.default_rng(7).standard_normal(3 * m.NP) * 1e-3
    x, res, h, resident = _device_solve(m, x0)
    assert resident > 0 and (groups is None or resident == groups), resident
    xr, info = restate.solve_krylov(m, x0=x0)
    assert res.error == info["error"] == (0 if maxit == 3000 else 3001)
    assert abs(res.iter - info["iter"]) <= max(3, 0.02 * info["iter"]), (res.iter, info["iter"])
    _same_start(h, info["history"])
    if maxit == 3000:
        r = m.B[:3 * m.N] - restate.matvec(m, x)
        assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
    # x after the same number of updates, or to the same residual
    assert np.linalg.norm(x - xr) <= 1e-6 * np.linalg.norm(xr)
    x2, res2, h2, launches = _device_solve(_with_external_node(m), np.concatenate([x0, np.zeros(3)]))
    assert launches == 0 and abs(res.iter - res2.iter) <= max(3, 0.02 * res2.iter)
    _same_start(h, h2)


@pytest.mark.parametrize("maxit", [1, 2, 49, 50, 51, 100])
def test_iteration_limit_and_residual_period(maxit):
    """NOCONV at MAXIT, on both sides of the iterations that recompute the residual (every 50)."""
    m = fa.gen_hex8(10, kind="lognormal", seed=4)
    m.set_iter(maxit)
    m.set_precond(3)
    m.set_resid(1e-14)
    x0 = np.random.default_rng(7).standard_normal(3 * m.NP) * 1e-3
    x, res, h, resident = _device_solve(m, x0)
    xr, info = restate.solve_krylov(m, x0=x0)
    assert resident > 0
    assert (res.iter, res.error) == (info["iter"], info["error"]) == (maxit + 1, 3001)
    _same_start(h, info["history"])
    # the recurrence carries a rounding unit of its largest entry per iteration; RESID is that
    # of the x that is returned, or of the recurrence that led to it
    r = m.B - restate.matvec(m, x)
    assert abs(np.linalg.norm(r) / np.linalg.norm(m.B) - res.resid) <= 1e-6 * res.resid + maxit * 1.1e-16 * h.max()
    if maxit <= 51:  # later iterates of the unconverged CG amplify a change of 1e-15 in x0 beyond that
        np.testing.assert_allclose(x, xr, rtol=0, atol=1e-6 * np.abs(xr).max())


def test_more_iterations_than_one_launch_and_new_values():
    """Two launches of the kernel (at most 512 iterations each), then other values on the
    same structure: the registers are filled from the present matrix."""
    import torch
    ctx = fa.DeviceContext()
    for seed in (1, 2):
        m = fa.gen_hex8(20, kind="lognormal", seed=seed)
        m.set_iter(5000)
        m.set_precond(3)
        m.set_resid(1e-10)
        ctx.load(m)
        b = torch.from_numpy(m.B).cuda()
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        res = ctx.solve_device(b.data_ptr(), x.data_ptr(), m.Iarray.copy(), m.Rarray)
        assert res.error == 0 and res.iter > 512 and ctx.info()["resident"] > 64, res.iter
        r = m.B - restate.matvec(m, x.cpu().numpy())
        assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
    ctx.close()


def test_rows_too_long_for_a_task_take_the_launches():
    m = random_system(240, deg=220, seed=3)  # four rows need more than 64 lanes of seven blocks
    m.set_iter(2000)
    m.set_precond(3)
    m.set_resid(1e-10)
    x, res, h, resident = _device_solve(m)
    assert resident == 0 and res.error == 0
    r = m.B - restate.matvec(m, x)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
