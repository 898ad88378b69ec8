"""The marching passes with non-temporal stores, which lattices beyond the
memory-side cache take, against those with plain stores: a lattice that repeats a
small one along z, so that it crosses the sizes of the rule (288 MB of state for
FIRE, in rows of a multiple of 64 bytes, 256 MB for Adam and Nesterov), while the
small one stays below.  Both hold a wall across x, whose sites the boundary pass
finishes in what the marching pass has stored, with one lane per site in both
lattices (more than 18,432 of them).

Adam and Nesterov advance every copy of a site by the same operations on the same
numbers: bit for bit.  FIRE's partial sums are added in another order: scalars agree
to roundings in FP64, below one rounding of Q per iteration."""
import numpy as np
import pytest

import pyoracle as po
import qmin
from test_gpu_parity import ALL, MULTI, ONE

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)
SMALL = (112, 97, 100)   # rows of 112 sites: a multiple of 64 bytes in both precisions
FIELDS = {"fire": 6, "adam": 4, "nesterov": 3}   # of five reals, that a pass touches
ITERATIONS = 6


def minimizer(name):
    return {"fire": lambda: qmin.FIRE(max_iter=ITERATIONS), "adam": lambda: qmin.Adam(dt=1e-3, max_iter=ITERATIONS),
            "nesterov": lambda: qmin.Nesterov(dt=1e-3, max_iter=ITERATIONS)}[name]()


def copies(name, precision):
    real = 8 if precision == qmin.QM_FP64 else 4
    per = 5 * FIELDS[name] * real * int(np.prod(SMALL))
    return int((288e6 if name == "fire" else 256e6) / per) + 1


def lattice(lz, precision, tile):
    g = qmin.Lattice(SMALL[0], SMALL[1], lz, precision=precision)
    g.set_tile(tile)
    g.set_zchunk(50)
    return g


@pytest.mark.parametrize("name", ["fire", "adam", "nesterov"])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
@pytest.mark.parametrize("tile,params", [(0, ONE), (0, ALL), (1, MULTI), (2, MULTI), (3, ONE)])
def test_nontemporal_stores_write_what_plain_ones_do(name, precision, tile, params):
    k = copies(name, precision)
    print("non-temporal stores: %s, precision %d, tile %d, %d copies" % (name, precision, tile, k), flush=True)
    f = qmin.LandauDeGennesLC(A, B, C, *params, semantics=1)
    small, big = lattice(SMALL[2], precision, tile), lattice(k * SMALL[2], precision, tile)
    small.random_init(17, S0)
    q0 = small.q()
    for g in (small, big):
        g.wall(0, 0, 1, 5.3, S0)
        assert g.n_boundary() > 18432
    big.set_field(qmin.FIELD_Q, np.tile(q0, (k, 1)))
    small.set_field(qmin.FIELD_Q, q0)
    for g in (small, big):
        minimizer(name).minimize(f, g)
    eps = 2.0 ** -52 if precision == qmin.QM_FP64 else 2.0 ** -23
    for which in (qmin.FIELD_Q, qmin.FIELD_V, qmin.FIELD_F):
        want, got = small.get_field(which), big.get_field(which).reshape(k, -1, 5)
        # FIRE: one rounding per iteration, of Q and v below 1; of F, whose stencils
        # add some thirty of Q with weights of up to 10, three hundred
        bound = 0 if name != "fire" else ITERATIONS * eps * (300 if which == qmin.FIELD_F else 1)
        for z in range(k):
            assert np.array_equal(got[z], want) if bound == 0 else np.abs(got[z] - want).max() <= bound, (which, z)
