"""Fields across the host boundary: whole lattices whose sites do not fill the
last work-group of the transposition, both precisions, and readers that overlap
in several threads."""
import threading

import numpy as np
import pytest

import pyoracle as po
import qmin

pytestmark = pytest.mark.gpu

A, B, C = po.rescaled_phase()
S0 = po.uniaxial_s0(A, B, C)


@pytest.mark.parametrize("shape", [(3, 3, 3), (16, 16, 1 + 2), (17, 31, 5), (64, 16, 9)])
@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_fields_round_trip(shape, precision):
    g = qmin.Lattice(*shape, precision=precision)
    rng = np.random.default_rng(shape[0])
    want = {}
    for which in (qmin.FIELD_Q, qmin.FIELD_V, qmin.FIELD_F):
        a = rng.normal(size=(g.n, 5))
        g.set_field(which, a)
        want[which] = a if precision == qmin.QM_FP64 else a.astype(np.float32).astype(np.float64)
    for which, a in want.items():
        assert np.array_equal(g.get_field(which), a)
    f = qmin.LandauDeGennesLC(A, B, C, 2.32)
    f.energy_density(g)
    g.defects(2)
    for which, a in want.items():
        assert np.array_equal(g.get_field(which), a)


def test_overlapping_readers():
    g = qmin.Lattice(70, 41, 33)
    g.random_init(5, S0)
    f = qmin.LandauDeGennesLC(A, B, C, 2.32)
    f.compute_forces(g)
    reads = [g.q, g.f, lambda: g.defects(0), lambda: g.defects(1), lambda: f.energy_density(g)]
    want = [r() for r in reads]
    bad = []

    def work(k):
        for _ in range(20):
            if not np.array_equal(reads[k](), want[k]):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(reads))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
