"""Energies of two forces taken on one lattice by two threads at once, and then
the forces of either: the operators that the lattice keeps are those of the
constants it has noted, whichever thread came last."""
import threading

import numpy as np
import pytest

import qmin
from test_gpu_parity import A, ALL, B, C, MULTI, build_pair

pytestmark = pytest.mark.gpu


def test_forces_after_overlapping_energies():
    _, g, first = build_pair((20, 18, 12), MULTI, 1, True)
    second = qmin.LandauDeGennesLC(A, B, C, *ALL, semantics=1)
    want = [f.compute_forces(g) for f in (first, second)]
    density = [f.energy_density(g) for f in (first, second)]
    bad = []

    def work(f, d):
        for _ in range(20):
            if not np.array_equal(f.energy_density(g), d):
                bad.append(d)

    for turn in range(60):
        threads = [threading.Thread(target=work, args=a) for a in zip((first, second), density)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
        order = (0, 1) if turn % 2 else (1, 0)
        for k in order:
            assert np.array_equal((first, second)[k].compute_forces(g), want[k]), (turn, k)
