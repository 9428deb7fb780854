"""GPU: the FP64 product below and above the 256 MB at which its matrix loads change
(csrc/kernels.hip), bitwise the restatement's (oracle/restate.c): the same operations in
the same order on the same values."""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import restate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,streamed", [(46, False), (53, True)])
def test_product_of_a_large_matrix(n, streamed):
    import torch
    m = fa.gen_hex8(n, kind="lognormal", seed=n)
    m.set_precond(3)
    ctx = fa.DeviceContext()
    ctx.load(m)
    assert (76 * ctx.info()["nslots"] > 256 << 20) == streamed
    x = np.random.default_rng(n).standard_normal(3 * m.NP)
    xt = torch.from_numpy(x).cuda()
    y = torch.full_like(xt, float("nan"))
    torch.cuda.synchronize()
    ctx.matvec_device(xt.data_ptr(), y.data_ptr(), 1)
    assert np.array_equal(y.cpu().numpy()[:3 * m.N], restate.matvec(m, x))
    ctx.close()
