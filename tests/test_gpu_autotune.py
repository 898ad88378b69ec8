"""The tile autotuner on small lattices, whose automatic pass goes by blocks: on
a fresh lattice with a tile or a z chunk set, whose first pass is then one that
has more partial sums than the set one's."""
import numpy as np
import pytest

import qmin
from test_gpu_parity import MULTI, ONE, build_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,params", [((64, 64, 64), ONE), ((50, 21, 7), MULTI)])
@pytest.mark.parametrize("tile,zchunk", [(0, 0), (-1, 16), (1, 4)])
def test_autotune_of_a_fresh_lattice_with_a_tile_set(shape, params, tile, zchunk):
    """The call succeeds (every pass it times fits the lattice's partial sums,
    which the library checks before each launch) and leaves the state alone;
    afterwards the lattice runs with the tile set again as an untuned one does."""
    print("autotune: shape %s, tile %d, z chunk %d" % (shape, tile, zchunk), flush=True)
    _, g, f = build_pair(shape, params, 1, True)
    q0 = g.q()
    g.set_tile(tile)
    g.set_zchunk(zchunk)
    g.autotune(f)
    assert np.array_equal(g.q(), q0)
    g.set_tile(tile)
    g.set_zchunk(zchunk)
    qmin.FIRE(max_iter=10).minimize(f, g)
    _, h, fh = build_pair(shape, params, 1, True)
    h.set_tile(tile)
    h.set_zchunk(zchunk)
    qmin.FIRE(max_iter=10).minimize(fh, h)
    assert np.array_equal(g.q(), h.q()) and np.array_equal(g.v(), h.v())


@pytest.mark.parametrize("precision", [qmin.QM_FP64, qmin.QM_FP32])
def test_autotune_keeps_the_tile_and_z_chunk_it_returns(precision):
    """They set on another lattice give the same run, sum for sum: other tiles, z
    chunks or blocks add the partial sums in another order."""
    runs = []
    for tune in (True, False):
        _, g, f = build_pair((40, 24, 20), MULTI, 1, True, precision=precision)
        if tune:
            tile, zchunk, ms = g.autotune(f)
            assert 0 <= tile <= 6 and zchunk in (0, 8, 16) and ms > 0
        else:
            g.set_tile(tile)
            g.set_zchunk(zchunk)
        m = qmin.FIRE(max_iter=40)
        m.set_trace(64)
        m.minimize(f, g)
        runs.append((m.trace(), g.q()))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
