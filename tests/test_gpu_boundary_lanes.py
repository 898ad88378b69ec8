"""Both forms of the boundary pass against the oracle: eight lanes per site (few
boundary sites) and one (many), with the same kinds of sites: walls, spheres of
both anchorings, corners between them, and bulk sites with one-sided neighbour
derivatives.  Forces and FIRE, Adam and Nesterov steps."""
import numpy as np
import pytest

import pyoracle as po
import qmin
from test_gpu_parity import ALL, MULTI, ONE, assert_forces_close

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)


def scene(shape, params, semantics, precision=qmin.QM_FP64):
    o, g = po.OracleSystem(*shape), qmin.Lattice(*shape, precision=precision)
    for s in (o, g):
        s.random_init(11, S0)
        s.wall(2, 0, 1, 5.3, S0)
        s.wall(2, shape[2] - 1, 0, 2.1, S0)
        s.sphere((shape[0] / 2, shape[1] / 3, 4.2), 2.6, 0, 3.0, S0)
        s.sphere((4.4, 6.1, 5.5), 1.8, 1, 1.5, S0)
    multi = params != ONE
    o.set_params(A, B, C, *params, multi=multi, semantics=semantics)
    return o, g, qmin.LandauDeGennesLC(A, B, C, *params, semantics=semantics)


# 16-site work-groups of eight lanes; more than 40960 sites take one lane each
@pytest.mark.parametrize("shape,many", [((20, 15, 9), False), ((160, 132, 9), True)])
@pytest.mark.parametrize("params", [ONE, MULTI, ALL])
@pytest.mark.parametrize("semantics", [0, 1])
def test_forces(shape, many, params, semantics):
    o, g, f = scene(shape, params, semantics)
    assert (g.n_boundary() > 40960) == many
    assert_forces_close(f.compute_forces(g), o.forces())


@pytest.mark.parametrize("shape", [(20, 15, 9), (160, 132, 9)])
def test_minimizers(shape):
    for make, run in ((lambda: qmin.FIRE(max_iter=6), lambda o: o.fire(max_iter=6)),
                      (lambda: qmin.Adam(dt=1e-3, max_iter=4), lambda o: o.adam(dt=1e-3, max_iter=4)),
                      (lambda: qmin.Nesterov(dt=1e-3, max_iter=4), lambda o: o.nesterov(dt=1e-3, max_iter=4))):
        o, g, f = scene(shape, MULTI, 1)
        make().minimize(f, g)
        run(o)
        np.testing.assert_allclose(g.q(), o.q(), rtol=0, atol=1e-12)


def test_stencils_follow_the_force_constants():
    """The composed stencils a lattice holds are those of the force it is used
    with: other constants, a change of precision and back."""
    o, g, f = scene((20, 15, 9), MULTI, 1)
    other = qmin.LandauDeGennesLC(A, B, C, *ALL, semantics=1)
    first = f.compute_forces(g)
    o.set_params(A, B, C, *ALL, multi=True, semantics=1)
    assert_forces_close(other.compute_forces(g), o.forces())
    assert np.array_equal(f.compute_forces(g), first)
    f.set_elastic(2.32, 0.7, 0.1)
    o.set_params(A, B, C, 2.32, 0.7, 0.1, 0.0, 0.0, multi=True, semantics=1)
    assert_forces_close(f.compute_forces(g), o.forces())
    g.set_precision(qmin.QM_FP32)
    f.compute_forces(g)
    g.set_precision(qmin.QM_FP64)
    o.set_q(g.q())
    assert_forces_close(f.compute_forces(g), o.forces())
