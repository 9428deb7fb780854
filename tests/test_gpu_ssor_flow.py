"""The FP32 SSOR application as one kernel (csrc/ssor_flow.hip) against the FP64
restatement of hecmw_precond_SSOR_33 (oracle/restate.c), at row lengths and sizes around
its groups of 8 blocks, its slices of 16 rows and its tickets of 8 slices.

With FP32 values every operation rounds to 6e-8, a row takes at most a few hundred of
them in sequence and the sweeps damp what they carry over (the systems are diagonally
dominant, or elastic with D an order above the rest): 3e-5 of the largest entry.  With
values that BF16 holds exactly, both formats are the same numbers, so the results are
equal to the last bit; and so is every repetition, whatever order the workgroups ran in.
"""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate
from tests.systems import random_system

pytestmark = pytest.mark.gpu

SYSTEMS = {
    "one_element": lambda: fa.gen_hex8(1),                      # a row per colour
    "few_rows": lambda: fa.gen_hex8(3, kind="lognormal", seed=2),
    "one_ticket_per_colour": lambda: fa.gen_hex8(11),
    "many_tickets": lambda: fa.gen_hex8(30, kind="lognormal", seed=2),
    "tet10": lambda: fa.gen_tet10(3, 2, 4, seed=1)[0],          # rows of more than 16 blocks
    "long_rows": lambda: random_system(900, deg=150, seed=3),   # many groups per row
    "odd_rows": lambda: random_system(777, deg=9, seed=5),
    "two_parts": lambda: random_system(500, deg=6, seed=6, components=2),
}


def _bf16(a):
    """The nearest value that BF16 holds."""
    u = a.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32)).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("sigma", [1.0, 1.35])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_ssor_f32_in_one_kernel(name, sigma):
    import torch
    m = SYSTEMS[name]()
    m.AL[:], m.AU[:] = _bf16(m.AL), _bf16(m.AU)
    m.set_precond(1)
    m.set_sigma_diag(sigma)
    ctx = fa.DeviceContext()
    ctx.load(m)
    r = np.random.default_rng(3).standard_normal(3 * m.NP).astype(np.float32)
    want = restate.precond(m, r.astype(np.float64))
    rt = torch.from_numpy(r).cuda()
    out = []
    for bf16 in (False, True, True):
        z = torch.full_like(rt, float("nan"))
        torch.cuda.synchronize()
        ctx.ssor_device(rt.data_ptr(), z.data_ptr(), 3, fp32=True, bf16=bf16)
        out.append(z.cpu().numpy()[:3 * m.N])
    ctx.close()
    err = np.abs(out[0] - want).max() / np.abs(want).max()
    assert err <= 3e-5, err
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[1], out[2])


def test_values_that_are_not_finite_pass_through():
    """A NaN in r (also one with the bits of the kernel's own mark) reaches the rows that
    depend on it and nothing waits for it; an infinity likewise."""
    import torch
    m = fa.gen_hex8(6, kind="lognormal", seed=2)
    m.set_precond(1)
    ctx = fa.DeviceContext()
    ctx.load(m)
    for bits in (0x7FFADEAD, 0x7FC00000, 0x7F800000):
        r = np.ones(3 * m.NP, np.float32)
        r[10] = np.array([bits], np.uint32).view(np.float32)[0]
        rt = torch.from_numpy(r).cuda()
        z = torch.zeros_like(rt)
        torch.cuda.synchronize()
        ms = ctx.ssor_device(rt.data_ptr(), z.data_ptr(), 1, fp32=True)
        z = z.cpu().numpy()
        assert not np.isfinite(z[9:12]).all() and ms < 1000.0
    ctx.close()
