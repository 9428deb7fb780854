"""The work users have this library do, as measurable cases.

A case is one call through the public Python entry points (which are the C ABI's,
one to one): whole solves through the drop-in host call and through device-resident
contexts, with each method and preconditioner, batched solves, and the two operators
(the matrix product and the SSOR application) by themselves.  Systems are the
repository's own synthetic models: HEX8 cubes with log-uniform stiffness (the
benchmark's material) or uniform material, and TET10 boxes.  The solves run to a
relative residual of 1e-10 (BiCGSTAB, whose residual says less about its error, 1e-11),
so that two correct solves agree to far better than single precision whatever order
their sums are taken in.
"""
import math

import numpy as np
import torch

import frontistr_amd as fa

RESID = 1e-10
MAXIT = 20000


def listed():
    return [
        # the first solve of a small test-sized model, as fistr1 calls it: host arrays, ordering,
        # factors and solve (the reference's solver tests have 100 to 600 nodes)
        {"name": "host_first_hex8_6", "kind": "host_first", "mesh": "lognormal", "n": 6},
        # a Newton step of an ordinary small model: new values on the known structure, numeric
        # set-up and solve, host arrays
        {"name": "host_newton_tet10_8", "kind": "host_newton", "mesh": "tet10", "n": 8},
        # plain SSOR-CG on resident systems: the 20^3 cube of the parity configuration, ...
        {"name": "cg_ssor_hex8_20", "kind": "cg_ssor", "mesh": "lognormal", "n": 20},
        # ... an ordinary odd-sized cube, and the largest
        {"name": "cg_ssor_hex8_41", "kind": "cg_ssor", "mesh": "uniform", "n": 41},
        {"name": "cg_ssor_hex8_72", "kind": "cg_ssor", "mesh": "lognormal", "n": 72},
        # block-Jacobi CG: the cheapest preconditioner, many short iterations
        {"name": "cg_diag_hex8_33", "kind": "cg_diag", "mesh": "lognormal", "n": 33},
        # BiCGSTAB with SSOR, the second Krylov method of the drop-in path, on quadratic tetrahedra
        {"name": "bicg_ssor_tet10_9", "kind": "bicg_ssor", "mesh": "tet10", "n": 9},
        # the mixed-precision two-level solve (deflation form) with its numeric set-up, the
        # fastest mode of the benchmark's headline system
        {"name": "two_level_hex8_48", "kind": "two_level", "mesh": "lognormal", "n": 48},
        # the same with the learned coarse modes, harvest and fit included
        {"name": "learned_hex8_30", "kind": "learned", "mesh": "lognormal", "n": 30},
        # several TET10 boxes with 16 load cases each in one batched solve
        {"name": "batch_tet10_6x16", "kind": "batch", "nsys": 6, "nrhs": 16, "dof_max": 30000,
         "sizes": 1},
        # the operators alone: FP64 product, FP32 SSOR application with BF16 couplings
        {"name": "matvec_hex8_72", "kind": "matvec", "mesh": "lognormal", "n": 72},
        {"name": "ssor_f32_hex8_60", "kind": "ssor_f32", "mesh": "lognormal", "n": 60},
    ]


# smallest and largest cube edge (HEX8 elements) per kind; a TET10 box has its nodes on the
# half-cell lattice, so the same node count at about half the cells (at most 14 of them: 27k nodes)
_RANGE = {"host_first": (4, 28), "host_newton": (4, 36), "cg_ssor": (5, 68), "cg_diag": (5, 44),
          "bicg_ssor": (5, 30), "two_level": (8, 64), "learned": (14, 44), "matvec": (6, 72),
          "ssor_f32": (6, 72)}


def draw(rng):
    kind = rng.choice(sorted(_RANGE) + ["batch"])
    if kind == "batch":
        return {"kind": kind, "nsys": rng.randint(2, 8), "nrhs": rng.choice([1, 3, 4, 8, 16]),
                "dof_max": int(math.exp(rng.uniform(math.log(3000), math.log(40000)))),
                "sizes": rng.randint(0, 999)}
    lo, hi = _RANGE[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    mesh = rng.choice(["lognormal", "uniform", "tet10"] if kind not in ("two_level", "learned") else
                      ["lognormal", "lognormal", "uniform"])
    if mesh == "tet10":
        n = min(14, max(2, n // 2))
    return {"kind": kind, "mesh": mesh, "n": n}


def _system(case, seed):
    """The assembled matrix, with loads (and for the lognormal cube stiffnesses) from the seed."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    if case["mesh"] == "tet10":
        m, _ = fa.gen_tet10(n, max(1, n - 1), n + 1, nrhs=1, seed=seed)
    else:
        m = fa.gen_hex8(n, kind=case["mesh"], seed=seed)
        m.B *= rng.uniform(0.5, 1.5, m.B.size)
    m.set_iter(MAXIT)
    m.set_resid(RESID if case["kind"] != "bicg_ssor" else 0.1 * RESID)
    return m


def _batch(case, seed):
    rng = np.random.default_rng(seed)
    mats, Bs, _ = fa.gen_tet10_batch(case["nsys"], case["nrhs"], dof_min=1000, dof_max=case["dof_max"],
                                     seed=case["sizes"])
    Bs = [B * rng.uniform(0.5, 1.5, B.shape) for B in Bs]
    mats[0].set_precond(3)
    mats[0].set_iter(MAXIT)
    mats[0].set_resid(RESID)
    return mats, Bs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mats, Bs = _batch(case, seed)
        return {"kind": kind, "solver": fa.BatchSolver(mats, Bs), "ia": mats[0].Iarray.copy(),
                "ra": mats[0].Rarray.copy(), "nsys": case["nsys"]}
    m = _system(case, seed)
    if kind in ("host_first", "host_newton"):
        return {"kind": kind, "m": m}
    m.set_precond(3 if kind == "cg_diag" else 1)
    m.set_method(2 if kind == "bicg_ssor" else 1)
    ctx = fa.DeviceContext()
    if kind in ("two_level", "learned"):
        m.set_mixed()
        m.set_coarse(1, deflation=True)
        ctx.set_coords(fa.hex8_coords(case["n"]))
    ctx.load(m)
    if kind == "learned":
        m.set_i(m.I_SOLVER_OPT, 2)
    # the two-level modes redo the numeric set-up on each solve, as a Newton step does; the
    # others keep the factors that the load made
    m.set_i(m.I_FLAG_NUMFACT, 1 if kind in ("two_level", "learned") else 0)
    m.set_i(m.I_FLAG_SYMBFACT, 0)
    dt = torch.float32 if kind == "ssor_f32" else torch.float64
    if kind in ("matvec", "ssor_f32"):
        b = torch.from_numpy(np.random.default_rng(seed).standard_normal(3 * m.NP)).to("cuda", dt)
    else:
        b = torch.from_numpy(m.B).to("cuda")
    x = torch.zeros(3 * m.NP, dtype=dt, device="cuda")
    torch.cuda.synchronize()
    return {"kind": kind, "ctx": ctx, "b": b, "x": x, "ia": m.Iarray.copy(), "ra": m.Rarray.copy()}


def run(state):
    kind = state["kind"]
    if kind == "batch":
        bs = state["solver"]
        bs.solve(state["ia"], state["ra"])
        return [bs.x(s) for s in range(state["nsys"])]
    if kind in ("host_first", "host_newton"):
        m = state["m"]
        m.X[:] = 0.0
        # Iarray 98 = 1: a new model; 97 = 2: new values, factors to be renewed
        m.set_i(m.I_FLAG_SYMBFACT, 1 if kind == "host_first" else 0)
        m.set_i(m.I_FLAG_NUMFACT, 2)
        fa.hecmw_solve_iterative(m)
        return m.X
    ctx, b, x = state["ctx"], state["b"], state["x"]
    if kind == "matvec":
        ctx.matvec_device(b.data_ptr(), x.data_ptr(), 1)
    elif kind == "ssor_f32":
        ctx.ssor_device(b.data_ptr(), x.data_ptr(), 1, fp32=True)
    else:
        x.zero_()
        torch.cuda.current_stream().synchronize()  # the context solves on a stream of its own
        ctx.solve_device(b.data_ptr(), x.data_ptr(), state["ia"], state["ra"])
    return x


def _counts(case):
    """(nodes, blocks) of a system."""
    n = case["n"]
    if case["mesh"] == "tet10":
        N = (2 * n + 1) * (2 * max(1, n - 1) + 1) * (2 * (n + 1) + 1)
        return N, 27.5 * N
    N = (n + 1) ** 3
    return N, (3 * n + 1) ** 3


def work(case):
    """Each iteration reads the blocks that its operators hold once (the SSOR factors and the
    matrix share their off-diagonal blocks) and its vectors; the iteration counts are those
    that the methods take to 1e-10 on these systems."""
    kind = case["kind"]
    if kind == "batch":
        nodes = case["nsys"] * math.sqrt(1000.0 * case["dof_max"]) / 3.0
        its = 35.0 * math.sqrt(case["dof_max"] / 1000.0) + 100.0
        per = 40.0 * 27.5 * nodes + case["nrhs"] * 12.0 * 8 * nodes
        return {"bytes": its * per, "flops": its * 18.0 * 27.5 * nodes * case["nrhs"]}
    N, nb = _counts(case)
    edge = N ** (1.0 / 3.0)
    w = 4 if kind in ("two_level", "learned", "ssor_f32") else 8
    its = {"host_first": 10.4 * edge + 20, "host_newton": 10.4 * edge + 20, "cg_ssor": 10.4 * edge + 20,
           "cg_diag": 29.0 * edge + 30, "bicg_ssor": 20.0 * edge, "two_level": 30 + 0.9 * edge,
           "learned": 90.0 + 0.6 * edge, "matvec": 1, "ssor_f32": 1}[kind]
    if kind == "ssor_f32":  # BF16 couplings
        per = 22.0 * nb + 9 * w * N + 2 * 3 * w * N
    else:
        per = (9 * w + 4.0) * nb + 2 * 3 * w * N
    if kind not in ("matvec", "ssor_f32"):
        per += 8 * 3 * w * N
    return {"bytes": its * per, "flops": its * 18.0 * nb}


def _ell(m):
    """Columns [N, w] and blocks [N, w, 3, 3] of the matrix rows, zero-padded, on the GPU."""
    N = m.N
    iL, iU = m.indexL[:N + 1].astype(np.int64), m.indexU[:N + 1].astype(np.int64)
    nl, nu = np.diff(iL), np.diff(iU)
    w = int((1 + nl + nu).max())
    cols = np.zeros((N, w), np.int64)
    vals = np.zeros((N, w, 9))
    cols[:, 0] = np.arange(N)
    vals[:, 0] = m.D.reshape(-1, 9)[:N]
    row = np.repeat(np.arange(N), nl)
    at = 1 + np.arange(iL[-1]) - np.repeat(iL[:-1], nl)
    cols[row, at] = m.itemL[:iL[-1]] - 1
    vals[row, at] = m.AL.reshape(-1, 9)[:iL[-1]]
    row = np.repeat(np.arange(N), nu)
    at = 1 + np.repeat(nl, nu) + np.arange(iU[-1]) - np.repeat(iU[:-1], nu)
    cols[row, at] = m.itemU[:iU[-1]] - 1
    vals[row, at] = m.AU.reshape(-1, 9)[:iU[-1]]
    return torch.from_numpy(cols).cuda(), torch.from_numpy(vals).cuda().reshape(N, w, 3, 3)


def _product(cols, vals, x):
    """A x for x [N, 3, k]."""
    y = torch.zeros_like(x)
    for j in range(cols.shape[1]):
        xj = x[cols[:, j]]
        for d in range(3):
            y += vals[:, j, :, d, None] * xj[:, d, None, :]
    return y


def _solution(m, B):
    """A^-1 B in FP64 (B [k, 3N]): scaled conjugate gradients to the rounding floor, restarted
    from the true residual."""
    cols, vals = _ell(m)
    b = torch.from_numpy(np.ascontiguousarray(B.reshape(len(B), m.N, 3).transpose(1, 2, 0))).cuda()
    dinv = 1.0 / torch.stack([vals[:, 0, d, d] for d in range(3)], 1)[:, :, None]
    x = torch.zeros_like(b)
    bn = (b * b).sum((0, 1))
    for tol in (1e-12, 1e-14):
        r = b - _product(cols, vals, x)
        z = dinv * r
        p, rz = z.clone(), (r * z).sum((0, 1))
        for it in range(MAXIT):
            q = _product(cols, vals, p)
            a = rz / (p * q).sum((0, 1)).clamp_min(1e-300)
            x += a * p
            r -= a * q
            if it % 50 == 49 and bool(((r * r).sum((0, 1)) <= tol * tol * bn).all()):
                break
            z = dinv * r
            new = (r * z).sum((0, 1))
            p = z + (new / rz.clamp_min(1e-300)) * p
            rz = new
    return x.permute(2, 0, 1).reshape(len(B), 3 * m.N)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ssor_f32":
        return None
    if kind == "batch":
        mats, Bs = _batch(case, seed)
        return [_solution(m, B) for m, B in zip(mats, Bs)]
    m = _system(case, seed)
    if kind == "matvec":
        cols, vals = _ell(m)
        x = torch.from_numpy(np.random.default_rng(seed).standard_normal(3 * m.NP)).cuda()
        return _product(cols, vals, x.reshape(m.N, 3, 1)).reshape(-1)
    return _solution(m, m.B[None])[0]
