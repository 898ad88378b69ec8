"""The force that an Adam or Nesterov run leaves when its tolerance stops it in one
of its first iterations, whose passes store it, or just after them: that of the same
run limited to as many."""
import numpy as np
import pytest

import qmin
from test_gpu_parity import MULTI, build_pair
from test_gpu_step_force import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["adam", "nesterov"])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("before", [0, 5])
def test_force_of_an_early_stop(name, precision, k, before):
    """before: iterations of the same minimizer in an earlier call."""
    shape = (37, 18, 9)
    out = []
    for tolerance in (False, True):
        _, g, f = build_pair(shape, MULTI, 1, True, precision=precision)
        m = make(name, fc=0.0, max_iter=before + k)
        if before:
            m.set_max_iterations(before)
            m.minimize(f, g)
        if tolerance:   # a minimizer whose tolerance the k-th iteration reaches, on the same state
            m = make(name, fc=fc, max_iter=1000)
        else:
            m = make(name, fc=0.0, max_iter=k)
            m.set_trace(k)
        m.minimize(f, g)
        if not tolerance:
            fm = m.trace()
            assert (np.diff(fm) < 0).all()
            fc = 1.000001 * fm[-1] if k == 1 else 0.5 * (fm[-1] + fm[-2])
        out.append((m.state()[0], g.q(), g.f()))
    assert out[0][0] == out[1][0] == k
    assert np.array_equal(out[0][1], out[1][1])
    tol = 1e-13 if precision == qmin.QM_FP64 else 1e-5
    np.testing.assert_allclose(out[1][2], out[0][2], rtol=0, atol=tol * np.abs(out[0][2]).max())
