"""What an ensemble run leaves on its lattices (Q, velocities, FIRE state) against
runs of the same lattices one by one, over two calls in a row and a single-lattice
run after them, for one lattice and for more than a wave of them."""
import numpy as np
import pytest

import qmin
from test_gpu_ensemble import A, B, C, SPECS, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
@pytest.mark.parametrize("count", [1, 6, 70])
def test_ensemble_leaves_the_lattices_as_single_runs_do(count, precision):
    specs = [(s[0], s[1] + 100 * k, s[2]) for k in range(12) for s in SPECS][:count]
    force = qmin.LandauDeGennesLC(A, B, C, 2.32, 0.0, 0.0, semantics=1)
    lats = [make(s, True, precision) for s in specs]
    alone = [make(s, True, precision) for s in specs]
    ens = qmin.Ensemble(lats)
    # order of the sums only: rounding, carried over 17 + 10 + 6 steps
    tol = 1e-11 if precision == qmin.QM_FP64 else 2e-6
    for n in (17, 10):
        its, _ = ens.fire_minimize(qmin.FIRE(fc=0.0, max_iter=n), force, 8)
        assert its.tolist() == [n] * count
        for x, y in zip(lats, alone):
            qmin.FIRE(fc=0.0, max_iter=n).minimize(force, y)
            np.testing.assert_allclose(x.q(), y.q(), rtol=0, atol=tol)
            np.testing.assert_allclose(x.v(), y.v(), rtol=0, atol=100 * tol)
    for x, y in zip(lats[:6], alone[:6]):
        for lat in (x, y):
            qmin.FIRE(fc=0.0, max_iter=6).minimize(force, lat)
        np.testing.assert_allclose(x.q(), y.q(), rtol=0, atol=tol)
        np.testing.assert_allclose(x.v(), y.v(), rtol=0, atol=100 * tol)
