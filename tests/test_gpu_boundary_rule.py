"""Which form of the boundary pass many and few sites take: an ensemble decides
by the sum of its lattices' boundary sites, so that its lattices take one lane per
site where each by itself takes eight."""
import numpy as np
import pytest

import pyoracle as po
import qmin
from test_gpu_parity import ALL, MULTI, ONE

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)


def lattices(precision):
    out = []
    for seed, shape in ((3, (84, 70, 9)), (4, (90, 75, 10)), (5, (61, 66, 8))):
        g = qmin.Lattice(*shape, precision=precision)
        g.random_init(seed, S0)
        g.wall(2, 0, 1, 5.3, S0)
        g.wall(2, shape[2] - 1, 0, 2.1, S0)
        out.append(g)
    return out


@pytest.mark.parametrize("params", [ONE, MULTI, ALL])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_ensemble_of_many_boundary_sites_follows_single_runs(params, precision):
    """Both forms compute the same sums in another order: ten iterations agree to
    some roundings of Q (below 1) per iteration."""
    f = qmin.LandauDeGennesLC(A, B, C, *params, semantics=1)
    single, batch = lattices(precision), lattices(precision)
    sites = [g.n_boundary() for g in single]
    assert max(sites) < 16384 and sum(sites) > 18432
    for g in single:
        qmin.FIRE(max_iter=10).minimize(f, g)
    qmin.Ensemble(batch).fire_minimize(qmin.FIRE(max_iter=10), f, 5)
    eps = 2.0 ** -52 if precision == qmin.QM_FP64 else 2.0 ** -23
    for a, b in zip(single, batch):
        np.testing.assert_allclose(b.q(), a.q(), rtol=0, atol=100 * eps)
