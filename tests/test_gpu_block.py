"""The block pass of small lattices (chosen automatically) against the marching
tiles, over lattices that its 16 x 4 x 4 blocks do not divide: forces bit for
bit, FIRE, Adam and Nesterov to rounding; and the oracle's forces."""
import numpy as np
import pytest

import pyoracle as po
import qmin
from test_gpu_parity import ALL, MULTI, ONE, assert_forces_close, build_pair

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (16, 4, 4), (17, 5, 9), (33, 3, 6), (50, 21, 7)]


def minimizer(name):
    return {"fire": lambda: qmin.FIRE(max_iter=20), "adam": lambda: qmin.Adam(dt=1e-3, max_iter=20),
            "nesterov": lambda: qmin.Nesterov(dt=1e-3, max_iter=20)}[name]()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("params", [ONE, MULTI, ALL])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_blocks_agree_with_tiles(shape, params, precision):
    objects = min(shape) > 5
    o, g, f = build_pair(shape, params, 1, objects, precision=precision)
    auto = f.compute_forces(g)
    g.set_tile(0)
    assert np.array_equal(auto, f.compute_forces(g))
    if precision == qmin.QM_FP64:
        assert_forces_close(auto, o.forces())
    for name in ("fire", "adam", "nesterov"):
        states = []
        for tile in (-1, 0):
            _, h, fh = build_pair(shape, params, 1, objects, precision=precision)
            h.set_tile(tile)
            minimizer(name).minimize(fh, h)
            states.append((h.q(), h.v()))
        tol = 1e-13 if precision == qmin.QM_FP64 else 0   # FP64 reduction rounding enters the FIRE mix, FP32 rounds it off
        np.testing.assert_allclose(states[0][0], states[1][0], rtol=0, atol=tol)
        np.testing.assert_allclose(states[0][1], states[1][1], rtol=0, atol=tol * 10)
