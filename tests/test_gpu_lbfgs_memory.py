"""Online L-BFGS over the sizes of its memory: one block of eight slots and
several, the recursion in LDS (up to 32 slots) and in memory, on a lattice whose
fields have an odd number of components; and calls that continue a run after
something else has computed forces on the lattice.  Against the oracle, with the
bound of the other L-BFGS traces (1e-9 relative)."""
import numpy as np
import pytest

import pyoracle as po
import qmin

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)


def pair(dims, precision=qmin.QM_FP64):
    o = po.OracleSystem(*dims)
    o.random_init(7, S0)
    o.sphere(tuple(d / 2 for d in dims), 2.3, 0, 2.0, S0)
    o.set_params(A, B, C, 2.32, 0.5, 0.3, 0.0, 0.0, multi=True, semantics=1)
    g = qmin.Lattice(*dims, precision=precision)
    g.random_init(7, S0)
    g.sphere(tuple(d / 2 for d in dims), 2.3, qmin.HOMEOTROPIC, 2.0, S0)
    return o, g, qmin.LandauDeGennesLC(A, B, C, 2.32, 0.5, 0.3)


@pytest.mark.parametrize("m,iterations", [(5, 14), (8, 20), (9, 24), (20, 45), (40, 60)])
def test_memory_sizes_match_oracle(m, iterations):
    o, g, f = pair((9, 11, 7))
    _, ref = o.lolbfgs(m=m, dt=2e-4, max_iter=iterations)
    ref = ref[:, 0] if ref.ndim == 2 else ref
    lb = qmin.LoLBFGS(m=m, dt=2e-4, fc=0.0, max_iter=iterations)
    lb.set_trace(iterations)
    lb.minimize(f, g)
    np.testing.assert_allclose(lb.trace(), ref[:iterations], rtol=1e-9)
    np.testing.assert_allclose(g.q(), o.q(), rtol=0, atol=1e-10)


@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_continued_run_keeps_its_direction(precision):
    """A run in two calls equals one in a single call, also if other forces were
    computed on the lattice between them: the direction and the forces it started
    from belong to the minimizer, y takes the lattice's forces."""
    _, a, f = pair((8, 9, 10), precision)
    _, b, _ = pair((8, 9, 10), precision)
    one = qmin.LoLBFGS(m=6, dt=2e-4, fc=0.0, max_iter=16)
    one.minimize(f, a)
    two = qmin.LoLBFGS(m=6, dt=2e-4, fc=0.0, max_iter=9)
    two.minimize(f, b)
    force = b.f()
    qmin.LandauDeGennesLC(A, B, C, 1.0).compute_forces(b)   # other forces on the same Q
    b.set_field(qmin.FIELD_F, force)
    two.set_max_iterations(16)
    two.minimize(f, b)
    assert one.state() == two.state()
    assert np.array_equal(a.q(), b.q())
