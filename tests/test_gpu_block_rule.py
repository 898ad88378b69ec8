"""Lattices beyond 131,072 sites on both sides of the line between the block pass
and the marching ones (short rows, flat lattices beside the FIRE pass that keeps
only Q and v): the automatic choice against a tile set by hand."""
import numpy as np
import pytest

import qmin
from test_gpu_parity import ALL, MULTI, ONE, build_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(17, 90, 90), (130, 129, 11), (128, 128, 32)])
@pytest.mark.parametrize("params", [ONE, MULTI, ALL])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_automatic_choice_agrees_with_a_set_tile(shape, params, precision):
    """Forces bit for bit; eight FIRE and eight Nesterov iterations to some roundings
    of Q (below 1) each: the FIRE pass that keeps only Q and v rounds its drift
    differently, and partial sums are added in another order."""
    out = []
    for tile in (-1, 0):
        _, g, f = build_pair(shape, params, 1, True, precision=precision)
        g.set_tile(tile)
        F = f.compute_forces(g)
        qmin.FIRE(max_iter=8).minimize(f, g)
        q = g.q()
        qmin.Nesterov(dt=1e-3, max_iter=8).minimize(f, g)
        out.append((F, q, g.q()))
    assert np.array_equal(out[0][0], out[1][0])
    eps = 2.0 ** -52 if precision == qmin.QM_FP64 else 2.0 ** -23
    np.testing.assert_allclose(out[0][1], out[1][1], rtol=0, atol=80 * eps)
    np.testing.assert_allclose(out[0][2], out[1][2], rtol=0, atol=160 * eps)
