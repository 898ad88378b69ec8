"""The allocation-free FIRE call on a lattice of many boundary sites: it takes
every lattice of up to 65,536 work-groups with 128 boundary sites counted as one,
which holds for both elastic models."""
import numpy as np
import pytest

import pyoracle as po
import qmin
from test_gpu_parity import MULTI, ONE

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)


@pytest.mark.parametrize("params", [ONE, MULTI])
@pytest.mark.parametrize("edge", [20, 1200])
def test_noalloc_fire_takes_many_boundary_sites(edge, params):
    """1200 x 1200 x 5 between two walls: 2.88 million boundary sites."""
    print("no-alloc FIRE between walls: edge %d" % edge, flush=True)
    f = qmin.LandauDeGennesLC(A, B, C, *params, semantics=1)
    out = []
    for noalloc in (False, True):
        g = qmin.Lattice(edge, edge, 5, precision=qmin.QM_FP32)
        g.random_init(5, S0)
        g.wall(2, 0, 1, 5.3, S0)
        g.wall(2, 4, 0, 2.0, S0)
        assert g.n_boundary() == 2 * edge * edge
        m = qmin.FIRE(max_iter=100)
        st = (m.run_iterations_noalloc if noalloc else m.run_iterations)(f, g, 3)
        out.append((st.forceMax, st.power, g.q(), g.v()))
    assert out[0][:2] == out[1][:2]
    assert np.array_equal(out[0][2], out[1][2]) and np.array_equal(out[0][3], out[1][3])
