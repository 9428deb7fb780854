"""oracle/ref.py where the reference's library is not built: the restatement answers what the
smoke solve and the learned modes' test ask of it."""
import numpy as np
import pytest

import frontistr_amd as fa
from oracle import ref, restate


def test_the_restatement_answers_where_the_library_is_not_built(monkeypatch, tmp_path):
    monkeypatch.setattr(ref, "LIB", str(tmp_path / "none.so"))
    monkeypatch.setattr(ref, "_lib", None)
    assert not ref.available()
    m = fa.gen_hex8(5, kind="lognormal", seed=1)
    m.set_iter(2000)
    x, info = ref.solve_krylov(m, nthreads=2)
    xr, want = restate.solve_krylov(m)
    assert np.array_equal(x, xr) and info["error"] == 0 and info["iter"] == want["iter"]
    assert np.array_equal(ref.matvec(m, x), restate.matvec(m, x))
    assert 0.0 < ref.rel_resid(m, x) <= 1e-8 * 1.0001
    with pytest.raises(RuntimeError):
        ref.precond(m, x)
