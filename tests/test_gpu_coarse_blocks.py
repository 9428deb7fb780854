"""GPU: the blocks of the coarse matrix E = Z^T A Z with few nodes per aggregate pair (a
wave per pair) and with many (a workgroup per pair) against numpy's product of the same A
and the Z of the library's own aggregates and offsets.  A block sums up to 1e5 products in
FP64 in another order: 1e-11 of the largest entry."""
import numpy as np
import pytest
from scipy import sparse

import frontistr_amd as fa

pytestmark = pytest.mark.gpu


def _csr(m):
    rows, cols, vals = [np.arange(m.N)], [np.arange(m.N)], [m.D.reshape(-1, 3, 3)[:m.N]]
    for idx, item, a in ((m.indexL, m.itemL, m.AL), (m.indexU, m.itemU, m.AU)):
        rows.append(np.repeat(np.arange(m.N), np.diff(idx[:m.N + 1])))
        cols.append(np.asarray(item) - 1)
        vals.append(a.reshape(-1, 3, 3))
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    i, j = np.meshgrid(np.arange(3), np.arange(3), indexing="ij")
    return sparse.coo_matrix((v.ravel(), ((3 * r[:, None, None] + i).ravel(), (3 * c[:, None, None] + j).ravel())),
                             shape=(3 * m.N, 3 * m.N)).tocsr()


@pytest.mark.parametrize("n,target,wave_per_pair", [(3, 8, True), (9, 64, True), (15, 8, False)])
def test_blocks_of_the_coarse_matrix(n, target, wave_per_pair):
    import torch
    m = fa.gen_hex8(n, kind="lognormal", seed=n)
    ctx = fa.DeviceContext()
    ctx.set_coords(fa.hex8_coords(n))
    mm = m.copy()
    mm.set_iter(3)
    mm.set_precond(1)
    mm.set_mixed(True)
    mm.set_coarse(target)
    ctx.load(mm)
    b = torch.tensor(mm.B, device="cuda:0")
    x = torch.zeros_like(b)
    ctx.solve_device(b.data_ptr(), x.data_ptr(), mm.Iarray, mm.Rarray)
    cs, entries = ctx.coarse(), ctx.info()["az_entries_symbolic"]
    ctx.close()
    na, agg, d = cs["n_agg"], cs["agg"], cs["dv"].astype(np.float64)
    assert (entries <= 64 * len(cs["pair_a"])) == wave_per_pair
    Z = np.zeros((m.N, 3, 6))
    Z[:, :, :3] = np.eye(3)
    Z[:, 0, 4], Z[:, 0, 5], Z[:, 1, 3], Z[:, 1, 5], Z[:, 2, 3], Z[:, 2, 4] = d[:, 2], -d[:, 1], -d[:, 2], d[:, 0], d[:, 1], -d[:, 0]
    rows = np.repeat(np.arange(3 * m.N), 6)
    cols = (6 * agg[:, None, None] + np.arange(6) + np.zeros((1, 3, 1), int)).ravel()
    Zs = sparse.csr_matrix((Z.ravel(), (rows, cols)), shape=(3 * m.N, 6 * na))
    E = (Zs.T @ (_csr(m) @ Zs)).toarray()
    for p, (a, c) in enumerate(zip(cs["pair_a"], cs["pair_b"])):
        err = np.abs(cs["Eblk"][p] - E[6 * a:6 * a + 6, 6 * c:6 * c + 6]).max()
        assert err <= 1e-11 * np.abs(E).max(), (p, a, c, err)
