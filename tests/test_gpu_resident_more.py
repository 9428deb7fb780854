"""The resident solves across the ends of their launches, beside each other on two threads, and
the systems that they leave to the launches; the FP32 sweeps with 512 workgroups."""
import threading

import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate
from tests import hip_shim
from tests.test_gpu_ssor_flow import _bf16

pytestmark = pytest.mark.gpu

EPS = 1.1e-16


def _context(m):
    ctx = fa.DeviceContext()
    ctx.load(m)
    ia = m.Iarray.copy()
    ia[m.I_FLAG_NUMFACT - 1] = ia[m.I_FLAG_SYMBFACT - 1] = 0
    return ctx, ia


def _abs_residual(m, x):
    """Largest rounding that one residual of x can hold, in units of EPS |b| and per operation."""
    a = m.copy()
    a.D, a.AL, a.AU = np.abs(m.D), np.abs(m.AL), np.abs(m.AU)
    return np.linalg.norm(restate.matvec(a, np.abs(x))) / np.linalg.norm(m.B)


# elements per edge, workgroups, Poisson's ratios: slow enough for 560 iterations, and not one of
# the systems near 1/2 on which BiCGSTAB breaks down (with the launches too, at others); 25^3
# gathers through the caches
@pytest.mark.parametrize("method,n,groups,nu", [
    (1, 6, 1, (0.499, 0.49999)), (1, 11, 32, (0.499, 0.49999)), (1, 25, 256, (0.499, 0.49999)),
    (2, 6, 1, (0.499, 0.49999)), (2, 11, 32, (0.49, 0.499)), (2, 25, 256, (0.45, 0.495))])
def test_a_second_launch_goes_on_where_the_first_ended(method, n, groups, nu):
    """A launch ends after 512 iterations.  560, ten (CG) and sixty (BiCGSTAB) after the last true
    residual: the recurrence residual that the second launch goes on with stays that of x.
    Rounding parts them by at most 81 operations a row and iteration on |A| |x| and on the
    largest residual so far."""
    import torch
    m = fa.gen_hex8(n, kind="lognormal", seed=2, numin=nu[0], numax=nu[1])
    m.set_precond(1)
    m.set_method(method)
    m.set_iter(560)
    m.set_resid(1e-14)
    ctx, ia = _context(m)
    b = torch.from_numpy(m.B).cuda()
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    res = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
    assert ctx.info()["resident"] == groups and (res.iter, res.error) == (561, 3001)
    h = ctx.history(560)
    ctx.close()
    x = x.cpu().numpy()
    true = np.linalg.norm(m.B - restate.matvec(m, x)) / np.linalg.norm(m.B)
    assert h[-1] == res.resid
    assert abs(true - res.resid) <= 60 * 81 * EPS * (_abs_residual(m, x) + h.max()), (true, res.resid)
    # nor does anything jump where the launch ends
    step = h[1:] / h[:-1]
    assert step[505:520].max() <= 10 * max(step[400:505].max(), step[520:].max())


def _upper_only(N, deg, seed):
    """Rows that read later rows, none of which reads them back."""
    rng = np.random.default_rng(seed)
    rows = [sorted(int(j) for j in rng.choice(N, deg, replace=False) if j > i) for i in range(N)]
    idx = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    item = np.array([j + 1 for r in rows for j in r], np.int32)
    return fa.HecMatrix(N, np.tile(np.eye(3).ravel() * 4.0, N), np.zeros(0), 0.1 * rng.standard_normal(9 * len(item)),
                        np.zeros(N + 1, np.int32), np.zeros(0, np.int32), idx, item, B=rng.standard_normal(3 * N))


def test_couplings_inside_a_colour_keep_the_launches():
    """The colouring of an unsymmetric profile leaves couplings inside a colour, for which a
    dataflow would wait (and give up after 20 s)."""
    import torch
    m = _upper_only(200, 5, 0)
    m.set_iter(5)
    m.set_precond(1)
    m.set_resid(1e-30)
    _, perm, iperm, ci = restate.ordering(m)
    colour = np.searchsorted(ci, iperm - 1, side="right")
    row = np.repeat(np.arange(m.N), np.diff(m.indexU))
    assert (colour[row] == colour[m.itemU - 1]).any()
    ctx, ia = _context(m)
    b = torch.from_numpy(m.B).cuda()
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    res = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
    assert ctx.info()["resident"] == 0 and np.isfinite(x.cpu().numpy()).all()
    r = torch.ones(3 * m.N, dtype=torch.float32, device="cuda")
    z = torch.zeros_like(r)
    torch.cuda.synchronize()
    ms = ctx.ssor_device(r.data_ptr(), z.data_ptr(), 1, fp32=True)
    assert ms < 1000.0 and np.isfinite(z.cpu().numpy()).all()
    # the next solve does not find that a wait was given up
    y = torch.zeros_like(b)
    torch.cuda.synchronize()
    again = ctx.solve_device(b.data_ptr(), y.data_ptr(), ia, m.Rarray)
    assert again.error == res.error
    ctx.close()


RECYCLED = """
a, b = fa.gen_hex8(8, kind="lognormal", seed=1), fa.gen_hex8(8, kind="lognormal", seed=2)
m = a.copy()
m.set_iter(3000)
m.set_resid(1e-10)
m.set_i(m.I_FLAG_NUMFACT, 2)
assert fa.hecmw_solve_iterative(m).error == 0
first = val("coop_calls").value
m.D[:], m.AL[:], m.AU[:] = b.D, b.AL, b.AU
m.X[:] = 0.0
m.set_i(m.I_FLAG_SYMBFACT, 0)
m.set_i(m.I_FLAG_NUMFACT, 1)
m.set_i(m.I_NRECYCLE, 0)
assert fa.hecmw_solve_iterative(m).error == 0 and m.get_i(m.I_NRECYCLE) == 1
second = val("coop_calls").value - first
r = m.B - restate.matvec(m, m.X)
print(first, second, np.linalg.norm(r) / np.linalg.norm(m.B))
"""


def test_recycled_factors_keep_the_launches(tmp_path):
    first, second, resid = hip_shim.run(tmp_path, RECYCLED)[-1].split()
    assert int(first) > 0 and int(second) == 0 and float(resid) <= 1.001e-10


def test_fp32_sweeps_with_512_workgroups():
    """More than 1280 slices of 16 rows a colour: two workgroups per CU.  Tolerances as for the
    other sizes (tests/test_gpu_ssor_flow.py)."""
    import torch
    m = fa.gen_hex8(70, kind="lognormal", seed=2)
    m.AL[:], m.AU[:] = _bf16(m.AL), _bf16(m.AU)
    m.set_precond(1)
    ctx, _ = _context(m)
    assert m.N // 16 // ctx.info()["ncolor"] // 8 >= 160
    r = np.random.default_rng(3).standard_normal(3 * m.NP).astype(np.float32)
    rt = torch.from_numpy(r).cuda()
    out = []
    for bf16 in (False, True, True):
        z = torch.full_like(rt, float("nan"))
        torch.cuda.synchronize()
        ctx.ssor_device(rt.data_ptr(), z.data_ptr(), 2, fp32=True, bf16=bf16)
        out.append(z.cpu().numpy())
    ctx.close()
    want = restate.precond(m, r.astype(np.float64))
    assert np.abs(out[0] - want).max() <= 3e-5 * np.abs(want).max()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[1], out[2])


def test_two_contexts_on_two_threads():
    """Resident kernels of two contexts, and FP32 sweeps, from two threads at once: every solve
    ends as alone, bit for bit, and stays resident (no wait ran out)."""
    import torch

    def system(n, method, precond):
        m = fa.gen_hex8(n, kind="lognormal", seed=2)
        m.set_iter(3000)
        m.set_resid(1e-10)
        m.set_method(method)
        m.set_precond(precond)
        return m

    jobs = [[system(19, 1, 1), system(12, 2, 1)], [system(15, 1, 3), system(27, 1, 1)]]
    state = [[(m, *_context(m), torch.from_numpy(m.B).cuda()) for m in pair] for pair in jobs]
    sweep = torch.ones_like(state[0][0][3], dtype=torch.float32)
    torch.cuda.synchronize()

    def solve(m, ctx, ia, b):
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        res = ctx.solve_device(b.data_ptr(), x.data_ptr(), ia, m.Rarray)
        return x.cpu().numpy(), res.iter, res.error, ctx.info()["resident"]

    def apply(ctx):
        z = torch.zeros_like(sweep)
        torch.cuda.synchronize()
        ctx.ssor_device(sweep.data_ptr(), z.data_ptr(), 1, fp32=True)
        return z.cpu().numpy()

    alone = [[solve(*s) for s in pair] for pair in state]
    z0 = apply(state[0][0][1])
    failed = []

    def run(k):
        try:
            for turn in range(6):
                for s, want in zip(state[k], alone[k]):
                    got = solve(*s)
                    assert got[2] == 0 and got[3] == want[3] > 0 and got[1] == want[1]
                    assert np.array_equal(got[0], want[0])
                if k == 0:
                    assert np.array_equal(apply(state[0][0][1]), z0)
        except BaseException as e:
            failed.append((k, repr(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for pair in state:
        for s in pair:
            s[1].close()
    assert not failed, failed
