"""The resident SSOR-CG and SSOR-BiCGSTAB kernels (csrc/resident.hip) against the plain-C
restatement of hecmw_solve_CG and hecmw_solve_BiCGSTAB (oracle/restate.c) and against the launch-per-colour solve, which a
system with an external node takes.

Both sides form the same sums in another order, so the residual histories differ by
rounding: about 1e-16 per operation, 1e3 operations deep and amplified by the
condition of these systems (up to 1e5) over the first iterations, hence 1e-8 on the
first fifteen.  (The entries are relative to |b|: one at the level of 1e-7 or below
holds rounding of 1e-16 |b| that is more than 1e-9 of it, and says nothing here.)
BiCGSTAB's polynomial amplifies rounding faster than CG's: five entries, and iteration
counts within the tenth that its other tests allow.  Solutions to a 1e-10 residual agree to 1e-6, the bar of every solve
here (the condition bounds the factor by 1e4).
"""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate
from tests.systems import random_system

pytestmark = pytest.mark.gpu


def _same_start(h, ref, most=15):
    k = min(most, len(h), len(ref))
    k = min([k] + [i for i in range(k) if ref[i] <= 1e-7])
    np.testing.assert_allclose(h[:k], ref[:k], rtol=1e-8)


def _with_external_node(m):
    """The same system with an external node that no row reads."""
    one = np.eye(3).ravel()
    m2 = fa.HecMatrix(m.N, np.concatenate([m.D, one]), m.AL, m.AU, np.append(m.indexL, m.NPL), m.itemL,
                      np.append(m.indexU, m.NPU), m.itemU, B=np.concatenate([m.B, np.zeros(3)]), NP=m.N + 1)
    m2.Iarray[:], m2.Rarray[:] = m.Iarray, m.Rarray
    return m2


def _device_solve(m, x0=None):
    import torch
    ctx = fa.DeviceContext()
    ctx.load(m)
    ia = m.Iarray.copy()
    ia[m.I_FLAG_NUMFACT - 1] = ia[m.I_FLAG_SYMBFACT - 1] = 0
    b = torch.from_numpy(m.B).cuda()
    x = torch.from_numpy(np.zeros(3 * m.NP) if x0 is None else x0).cuda()
    torch.cuda.synchronize()
    res = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
    return x.cpu().numpy(), res, ctx.history(max(1, min(res.iter, m.get_i(m.I_ITER)))), ctx.info()["resident"]


# name: system, workgroups that the rule picks
SYSTEMS = {
    "one_element": (lambda: fa.gen_hex8(1), 1),                     # a row per colour
    "one_group": (lambda: fa.gen_hex8(6, kind="lognormal", seed=2), 1),
    "just_past_one_group": (lambda: fa.gen_hex8(7, kind="lognormal", seed=2), 32),
    "past_one_group": (lambda: fa.gen_hex8(10), 32),
    "tet10_small": (lambda: fa.gen_tet10(3, 2, 4, seed=1)[0], 1),
    "grid_128": (lambda: fa.gen_hex8(15, kind="lognormal", seed=2), 128),
    "grid_256": (lambda: fa.gen_hex8(25), 256),
    "long_rows": (lambda: random_system(900, deg=150, seed=3), None),    # more than 128 blocks in a row
    "odd_rows": (lambda: random_system(777, deg=9, seed=5), 32),
    "odd_rows_one_group": (lambda: random_system(433, deg=9, seed=5), 1),
    "two_parts": (lambda: random_system(500, deg=6, seed=6, components=2), 32),
}


@pytest.mark.parametrize("sigma", [1.0, 1.35])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_resident_cg_matches_the_restatement(name, sigma):
    make, groups = SYSTEMS[name]
    m = make()
    m.set_iter(3000)
    m.set_precond(1)
    m.set_resid(1e-10)
    m.set_sigma_diag(sigma)
    x, res, h, resident = _device_solve(m)
    assert resident > 0 and (groups is None or resident == groups), resident
    xr, info = restate.solve_krylov(m)
    assert res.error == 0 and info["error"] == 0
    assert abs(res.iter - info["iter"]) <= 2, (res.iter, info["iter"])
    assert res.resid <= 1e-10
    r = m.B[:3 * m.N] - restate.matvec(m, x)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
    assert np.linalg.norm(x - xr) <= 1e-6 * np.linalg.norm(xr)
    _same_start(h, info["history"])
    x2, res2, h2, launches = _device_solve(_with_external_node(m))
    assert launches == 0 and abs(res.iter - res2.iter) <= 2
    _same_start(h, h2)


@pytest.mark.parametrize("maxit", [1, 2, 49, 50, 51, 100])
@pytest.mark.parametrize("n", [4, 11])
def test_iteration_limit_and_residual_period(n, maxit):
    """NOCONV at MAXIT, on both sides of the iterations that recompute the residual (every
    50): the same ITER, error and history as the restatement, x after MAXIT updates."""
    m = fa.gen_hex8(n, kind="lognormal", seed=4)
    m.set_iter(maxit)
    m.set_precond(1)
    m.set_resid(1e-14)
    x0 = np.random.default_rng(7).standard_normal(3 * m.NP) * 1e-3
    x, res, h, resident = _device_solve(m, x0)
    xr, info = restate.solve_krylov(m, x0=x0)
    assert resident > 0
    assert (res.iter, res.error) == (info["iter"], info["error"])
    _same_start(h, info["history"])
    if maxit <= 51:
        # the recurrence carries a rounding unit of its largest entry per iteration
        np.testing.assert_allclose(h, info["history"], rtol=1e-5, atol=maxit * 1.1e-16 * h.max())
        assert np.linalg.norm(x - xr) <= 1e-6 * np.linalg.norm(xr)


@pytest.mark.parametrize("sigma", [1.0, 1.35])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_resident_bicgstab_matches_the_restatement(name, sigma):
    make, groups = SYSTEMS[name]
    m = make()
    m.set_iter(3000)
    m.set_method(2)
    m.set_precond(1)
    m.set_resid(1e-10)
    m.set_sigma_diag(sigma)
    x, res, h, resident = _device_solve(m)
    assert resident > 0 and (groups is None or resident == groups), resident
    xr, info = restate.solve_krylov(m)
    assert res.error == 0 and info["error"] == 0
    assert abs(res.iter - info["iter"]) <= 2 + 0.1 * info["iter"], (res.iter, info["iter"])
    assert res.resid <= 1e-10
    r = m.B[:3 * m.N] - restate.matvec(m, x)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
    assert np.linalg.norm(x - xr) <= 1e-6 * np.linalg.norm(xr)
    _same_start(h, info["history"], 5)
    x2, res2, h2, launches = _device_solve(_with_external_node(m))
    assert launches == 0
    _same_start(h, h2, 5)


@pytest.mark.parametrize("maxit", [1, 2, 99, 100, 101])
def test_bicgstab_iteration_limit_and_residual_period(maxit):
    """NOCONV at MAXIT, on both sides of the iteration that recomputes the residual (every 100)."""
    m = fa.gen_hex8(11, kind="lognormal", seed=4)
    m.set_iter(maxit)
    m.set_method(2)
    m.set_precond(1)
    m.set_resid(1e-14)
    x0 = np.random.default_rng(7).standard_normal(3 * m.NP) * 1e-3
    x, res, h, resident = _device_solve(m, x0)
    _, info = restate.solve_krylov(m, x0=x0)
    assert resident > 0
    assert (res.iter, res.error) == (info["iter"], info["error"]) == (maxit + 1, 3001)
    _same_start(h, info["history"], 5)
    # RESID is the residual of the x that is returned
    r = m.B - restate.matvec(m, x)
    assert abs(np.linalg.norm(r) / np.linalg.norm(m.B) - res.resid) <= 1e-6 * res.resid + maxit * 1.1e-16 * h.max()


def test_method_change_on_one_context():
    """CG, BiCGSTAB and CG again on the same context: the row records change layout."""
    import torch
    m = fa.gen_hex8(9, kind="lognormal", seed=3)
    m.set_iter(2000)
    m.set_precond(1)
    m.set_resid(1e-10)
    ctx = fa.DeviceContext()
    ctx.load(m)
    b = torch.from_numpy(m.B).cuda()
    out = []
    for method in (1, 2, 1):
        ia = m.Iarray.copy()
        ia[m.I_METHOD - 1] = method
        ia[m.I_FLAG_NUMFACT - 1] = ia[m.I_FLAG_SYMBFACT - 1] = 0
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        res = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
        assert res.error == 0 and ctx.info()["resident"] > 0
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0], out[2])
    assert np.linalg.norm(out[1] - out[0]) <= 1e-6 * np.linalg.norm(out[0])


def test_more_iterations_than_one_launch():
    """A solve that takes two launches of the kernel (at most 512 iterations each)."""
    m = fa.gen_hex8(56, kind="lognormal", seed=1)
    m.set_iter(20000)
    m.set_precond(1)
    m.set_resid(1e-10)
    x, res, h, resident = _device_solve(m)
    assert resident > 0 and res.error == 0 and res.iter > 512, res.iter
    r = m.B - restate.matvec(m, x)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)
    x2, res2, _, launches = _device_solve(_with_external_node(m))
    assert launches == 0 and abs(res.iter - res2.iter) <= 2
    x2 = x2[:3 * m.N]
    assert np.linalg.norm(x - x2) <= 1e-6 * np.linalg.norm(x2)


def test_new_values_reach_the_packed_copy():
    """A second matrix on the same structure, through the host entry point."""
    for seed in (1, 2):
        m = fa.gen_hex8(9, kind="lognormal", seed=seed)
        m.set_iter(2000)
        m.set_resid(1e-10)
        m.set_i(m.I_FLAG_SYMBFACT, 1 if seed == 1 else 0)
        m.set_i(m.I_FLAG_NUMFACT, 2)
        res = fa.hecmw_solve_iterative(m)
        xr, info = restate.solve_krylov(m)
        assert res.error == 0 and abs(res.iter - info["iter"]) <= 2
        assert np.linalg.norm(m.X - xr) <= 1e-6 * np.linalg.norm(xr)


def test_recycled_preconditioner_takes_the_launches():
    """With factors of older values the sweeps cannot give A z: the launch-per-colour solve
    runs, and its solution solves the new system."""
    import torch
    a, b = fa.gen_hex8(8, kind="lognormal", seed=1), fa.gen_hex8(8, kind="lognormal", seed=2)
    m = a.copy()
    m.set_iter(3000)
    m.set_resid(1e-10)
    m.set_i(m.I_FLAG_NUMFACT, 2)
    assert fa.hecmw_solve_iterative(m).error == 0
    m.D[:], m.AL[:], m.AU[:] = b.D, b.AL, b.AU
    m.X[:] = 0.0
    m.set_i(m.I_FLAG_SYMBFACT, 0)
    m.set_i(m.I_FLAG_NUMFACT, 1)
    m.set_i(m.I_NRECYCLE, 0)
    assert fa.hecmw_solve_iterative(m).error == 0
    assert m.get_i(m.I_NRECYCLE) == 1
    r = m.B - restate.matvec(m, m.X)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(m.B)


@pytest.mark.parametrize("what", ["rows over 256 blocks", "unsymmetric profile"])
def test_systems_that_keep_the_launches(what):
    if what == "rows over 256 blocks":
        m = random_system(700, deg=420, seed=8)
    else:
        # node 2 reads node 1, not the other way round, in a chain of such couplings
        N = 40
        D = np.tile(np.eye(3).ravel() * 4.0, N)
        iL = np.concatenate([[0], np.arange(N)]).astype(np.int32)
        AL = np.tile((0.1 * np.eye(3)).ravel(), N - 1)
        m = fa.HecMatrix(N, D, AL, np.zeros(0), iL, np.arange(1, N, dtype=np.int32), np.zeros(N + 1, np.int32),
                         np.zeros(0, np.int32), B=np.ones(3 * N))
        m.set_iter(5)
    m.set_precond(1)
    if what == "rows over 256 blocks":
        m.set_iter(500)
    x, res, _, resident = _device_solve(m)
    assert np.isfinite(x).all()
    if what == "rows over 256 blocks":
        assert resident == 0 and res.error == 0
        xr, info = restate.solve_krylov(m)
        assert np.linalg.norm(x - xr) <= 1e-6 * np.linalg.norm(xr)


def test_nan_right_hand_side_ends_the_solve():
    m = fa.gen_hex8(6)
    m.set_iter(200)
    m.B[4] = np.nan
    x, res, _, resident = _device_solve(m)
    _, info = restate.solve_krylov(m)
    assert resident > 0 and res.error == info["error"]
