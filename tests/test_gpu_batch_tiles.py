"""Batched solves with tiles of 16, 32, 64 and 128 rows (csrc/batch.hip picks them by the
rows of the batch): the FP64 product is bitwise the restatement's SpMV (oracle/restate.c)
whatever the tiles, the FP32 one within its rounding (2e-6 in the norm, as in the other
batch tests), and a solve reaches its FP64 residual for every system, also for one that
ends in a partial tile and one smaller than a tile."""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate

pytestmark = pytest.mark.gpu


# nodes per edge minus one of the largest system -> rows per tile on 256 CUs: 6 tiles per CU
@pytest.mark.parametrize("n,rows_per_tile", [(3, 16), (29, 32), (37, 64), (47, 128)])
def test_tiles_by_batch_size(n, rows_per_tile):
    mats = [fa.gen_hex8(n, kind="lognormal", seed=n), fa.gen_hex8(1), fa.gen_tet10(2, 3, 2, seed=1)[0]]
    rng = np.random.default_rng(n)
    Bs = [rng.standard_normal((2, 3 * m.N)) for m in mats]
    bs = fa.BatchSolver(mats, Bs)
    info = bs.info()
    assert info["tiles"] == sum(-(-m.N // rows_per_tile) for m in mats)
    Y64, Y32 = bs.spmm(Bs, fp64=True), bs.spmm(Bs, fp64=False)
    for m, X, y64, y32 in zip(mats, Bs, Y64, Y32):
        for k in range(2):
            y = restate.matvec(m, X[k])
            assert np.array_equal(y64[k], y)
            assert np.linalg.norm(y32[k] - y) <= 2e-6 * np.linalg.norm(y)
    p = fa.gen_hex8(1)
    p.set_iter(5000)
    p.set_precond(3)
    bs.solve(p.Iarray.copy(), p.Rarray.copy())
    for s, m in enumerate(mats):
        x = np.asarray(bs.x(s))
        for k in range(2):
            r = Bs[s][k] - restate.matvec(m, x[k])
            assert np.linalg.norm(r) <= 1.001e-8 * np.linalg.norm(Bs[s][k])
    bs.close()


def test_instances_that_stop_at_different_times():
    """A zero column, NOCONV for all others at MAXIT 6 (ITER 7), then a solve to the end on the
    same loaded batch, whose instances converge in different iterations, one system long
    before the others: every solution within 1e-6 of the restatement's DIAG-CG."""
    mats = [fa.gen_hex8(1), fa.gen_hex8(9, kind="lognormal", seed=2), fa.gen_tet10(4, 2, 3, seed=1)[0], fa.gen_hex8(5)]
    rng = np.random.default_rng(3)
    Bs = [rng.standard_normal((3, 3 * m.N)) for m in mats]
    Bs[1][2][:] = 0.0
    bs = fa.BatchSolver(mats, Bs)
    p = fa.gen_hex8(1)
    p.set_precond(3)
    p.set_iter(6)
    it, er, rs, _ = bs.solve(p.Iarray.copy(), p.Rarray.copy())
    live = np.ones_like(er, dtype=bool)
    live[1, 2] = False
    assert np.all(er[live] == 3001) and np.all(it[live] == 7)
    assert it[1, 2] == 1 and er[1, 2] == 0 and np.all(bs.x(1)[2] == 0.0)
    p.set_iter(5000)
    it, er, rs, _ = bs.solve(p.Iarray.copy(), p.Rarray.copy())
    assert np.all(er == 0) and np.all(rs <= 1e-8) and it[1, 2] == 1
    for s, m in enumerate(mats):
        X = bs.x(s)
        for k in range(3):
            mk = m.copy()
            mk.B[:] = Bs[s][k]
            mk.set_precond(3)
            mk.set_iter(5000)
            if not live[s, k]:
                continue
            xr, info = restate.solve_krylov(mk)
            assert info["error"] == 0 and it[s, k] <= 1.3 * info["iter"] + 10
            assert np.linalg.norm(X[k] - xr) <= 1e-6 * np.linalg.norm(xr)
    bs.close()


def test_tuned_shapes_belong_to_their_tiles(tmp_path, monkeypatch):
    """A saved winner from other tiles (here a line without any) stays in the file but is not
    taken; the winner that the load finds is, by the next one."""
    import torch
    path = tmp_path / "tune.txt"
    monkeypatch.setenv("HECMW33_TUNE_CACHE", str(path))
    m = fa.gen_hex8(6)
    B = np.random.default_rng(1).standard_normal((1, 3 * m.N))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    old = "gfx950 %d %d %d lpr64_rpl1_u1 lpr16_rpl1_u1" % (cus, round((m.N + m.NPL + m.NPU) / m.N), int(np.log2(m.N)))
    path.write_text(old + "\n")
    for cached in (False, True):
        bs = fa.BatchSolver([m], [B])
        assert bs.info()["tune_cached"] == cached
        bs.close()
    lines = path.read_text().strip().splitlines()
    assert old in lines and len(lines) == 2 and any(l.startswith("gfx950-t16 ") for l in lines)
