"""FIRE on small lattices, where each pass begins with the previous iteration's
scalar step, against the marching tiles with a launch of its own for it: runs
shorter than, as long as and longer than one queued batch, continued runs, and a
tolerance reached within a batch."""
import numpy as np
import pytest

import qmin
from test_gpu_parity import MULTI, ONE, build_pair

pytestmark = pytest.mark.gpu

SHAPE = (17, 9, 11)


def run(params, precision, tile, counts, fc=0.0):
    _, g, f = build_pair(SHAPE, params, 1, True, precision=precision)
    g.set_tile(tile)
    out = []
    m = qmin.FIRE(fc=fc)
    for n in counts:
        s = m.run_iterations(f, g, n)
        out.append((s.iterations, s.forceMax, s.deltaT, s.alpha))
    return out, g.q(), g.v()


@pytest.mark.parametrize("params", [ONE, MULTI])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
@pytest.mark.parametrize("counts", [(1,), (2,), (3,), (1, 2, 4), (256,), (257,), (300, 5)])
def test_chained_runs_agree_with_separate_launches(params, precision, counts):
    a, qa, va = run(params, precision, -1, counts)
    b, qb, vb = run(params, precision, 0, counts)
    assert [x[0] for x in a] == [x[0] for x in b]
    rtol = 1e-6 if precision == qmin.QM_FP64 else 1e-3
    # the sums' order differs by rounding, which a trajectory of some hundred
    # steps carries on; a step taken twice, left out or with old scalars is 1e-5 and more
    tol = 1e-10 if precision == qmin.QM_FP64 else 1e-5
    np.testing.assert_allclose([x[1:] for x in a], [x[1:] for x in b], rtol=rtol, atol=tol)
    np.testing.assert_allclose(qa, qb, rtol=0, atol=tol)
    np.testing.assert_allclose(va, vb, rtol=0, atol=100 * tol)


@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_a_tolerance_reached_within_a_batch_ends_both_at_the_same_iteration(precision):
    trace, _, _ = run(ONE, precision, 0, tuple([1] * 40))
    cutoff = 0.5 * (trace[20][1] + trace[21][1])
    out = []
    for tile in (-1, 0):
        _, g, f = build_pair(SHAPE, ONE, 1, True, precision=precision)
        g.set_tile(tile)
        s = qmin.FIRE(fc=cutoff, max_iter=200).minimize(f, g)
        out.append((s.iterations, s.converged, g.q()))
    assert out[0][:2] == out[1][:2] and out[0][1] and out[0][0] < 200
    np.testing.assert_allclose(out[0][2], out[1][2], rtol=0, atol=1e-10 if precision == qmin.QM_FP64 else 1e-5)
