"""Grids of thousands of levels: the pass keeps three coefficients a level in LDS beside its tiles, so its tall FP64
tiles do not fit there.  The height that the library takes by itself has to, where the ranking alone would not."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from tests import decks

pytestmark = pytest.mark.gpu


# 16 x 16 cells: 4, 3, 3 and 2 tiles of 8, 10, 11 and 12 rows a slot.  With 100 slots 12 rows alone come in one round
# of 256 workgroups; up to 3157 levels they fit.
@pytest.mark.parametrize("levels,rows", [(3157, 12), (3158, 8), (4040, 8)])
def test_default_height_fits(levels, rows, monkeypatch):
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    st = decks.small_setup(T, nx=12, ny=12, nz=levels, pad=(1, 1))
    st.Az1 = st.Az2 = 0
    gi = T.grid_info(st)
    assert (gi.L, gi.M, gi.N) == (16, 16, levels)
    cond = decks.layered_cond((gi.N, gi.M, gi.L), T.grid_arrays(st)["Z"][:, None, None] * np.ones((1, gi.M, gi.L)))
    with T.Context(st, cond, T.FP64) as c:
        c.set_receivers(T.make_rxtime(0.02, 0.25, 8, 1, (1, 1, 1, 1, 1, 1)), np.array([[0.0, 0.0, 200.0]]))
        c.set_transmitters([T.make_tx(1, 100.0, 2.0 * q - 100.0, 0.0, 150.0, [1]) for q in range(100)])
        c.set_graph(0)
        c.begin(0, 100)
        assert c.pair_info()[0] == rows
        c.step(12)
        assert c.pair_info()[2] == 6
        got = [c.get(T.EX, q) for q in (0, 99)]
        c.set_pairs(0)
        c.begin(0, 100)
        c.step(12)
        for q, g in zip((0, 99), got):
            assert np.any(g) and np.array_equal(g, c.get(T.EX, q))
