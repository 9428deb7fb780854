"""GPU: the factorization and inverse of the coarse matrix E in blocks of 64 (chol.hip):
E^-1 against numpy's inverse of the same E at orders below, at and just above a multiple
of the block, with bands of one block, of several and of the whole matrix; and the
refusal of an E that is not positive definite, in the first block and in the last."""
import numpy as np
import pytest

import frontistr_amd as fa

pytestmark = pytest.mark.gpu


def _solve(m, coords, target, maxit):
    import torch
    ctx = fa.DeviceContext()
    ctx.set_coords(coords)
    mm = m.copy()
    mm.set_iter(maxit)
    mm.set_precond(1)
    mm.set_mixed(True)
    mm.set_coarse(target)
    ctx.load(mm)
    b = torch.tensor(mm.B, device="cuda:0")
    x = torch.zeros_like(b)
    r = ctx.solve_device(b.data_ptr(), x.data_ptr(), mm.Iarray, mm.Rarray)
    return ctx, r


# (elements per edge, aggregates aimed at) -> orders 48 (one block, padded), 162 (three, padded),
# 384 (six, no padding), 750 and 1296 (bands narrower than E)
@pytest.mark.parametrize("n,target,order", [(4, 8, 48), (8, 27, 162), (9, 64, 384), (13, 216, 750), (18, 512, 1296)])
def test_inverse_of_the_coarse_matrix(n, target, order):
    m = fa.gen_hex8(n, kind="lognormal", seed=n)
    ctx, r = _solve(m, fa.hex8_coords(n), target, 5000)
    assert r.error == 0
    cs = ctx.coarse()
    W, f64 = ctx.coarse_inverse()
    ctx.close()
    na, pa, pb, Eb = cs["n_agg"], cs["pair_a"], cs["pair_b"], cs["Eblk"]
    assert not f64 and 6 * na == order and W.shape == (order, order)
    E = np.zeros((order, order))
    for p in range(len(pa)):
        E[6 * pa[p]:6 * pa[p] + 6, 6 * pb[p]:6 * pb[p] + 6] = Eb[p]
    assert np.linalg.cond(E) < 1e8  # so that FP64 factors leave FP32 rounding of the copy as the error
    Ei = np.linalg.inv(E)
    err = np.abs(W.astype(np.float64) - Ei).max() / np.abs(Ei).max()
    assert err <= 2.0 ** -23, err
    assert np.array_equal(W, W.T)


@pytest.mark.parametrize("where", ["all", "last"])
def test_indefinite_coarse_matrix_is_refused(where):
    n = 8
    m = fa.gen_hex8(n, kind="lognormal", seed=1)
    if where == "all":
        m.D[:] = -m.D
        m.AL[:] = -m.AL
        m.AU[:] = -m.AU
    else:  # the last corner node only: the rows before it still eliminate
        m.D.reshape(-1, 9)[-1] *= -1e3
    ctx, _ = _solve(m, fa.hex8_coords(n), 27, 3)
    assert ctx.info()["coarse"] == -1
    ctx.close()
