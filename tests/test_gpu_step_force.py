"""The force an Adam or Nesterov run leaves on the lattice, that of the Q before
its last update, whether the run's limit or its tolerance ended it: a run that
its tolerance stops after k iterations against one limited to k, for odd and even
k, runs short enough to store every force, and lattices of blocks and of tiles."""
import numpy as np
import pytest

import qmin
from test_gpu_parity import MULTI, build_pair

pytestmark = pytest.mark.gpu


def make(name, **kw):
    return qmin.Adam(dt=1e-3, **kw) if name == "adam" else qmin.Nesterov(dt=1e-3, **kw)


@pytest.mark.parametrize("name", ["adam", "nesterov"])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
@pytest.mark.parametrize("tile", [-1, 2])
@pytest.mark.parametrize("k", [2, 7, 10])
def test_force_of_the_last_iteration(name, precision, tile, k):
    shape = (37, 18, 9)
    _, a, f = build_pair(shape, MULTI, 1, True, precision=precision)
    _, b, _ = build_pair(shape, MULTI, 1, True, precision=precision)
    for g in (a, b):
        g.set_tile(tile)
    limited = make(name, fc=0.0, max_iter=k)
    limited.set_trace(k)
    limited.minimize(f, a)
    fm = limited.trace()
    assert (np.diff(fm) < 0).all()   # so that a tolerance can pick the k-th iteration
    stopped = make(name, fc=0.5 * (fm[-1] + fm[-2]), max_iter=1000)
    stopped.minimize(f, b)
    assert stopped.state()[0] == k
    assert np.array_equal(a.q(), b.q())
    tol = 1e-13 if precision == qmin.QM_FP64 else 1e-5
    np.testing.assert_allclose(b.f(), a.f(), rtol=0, atol=tol * np.abs(a.f()).max())
