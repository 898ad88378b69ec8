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
