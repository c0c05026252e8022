"""The two-step pass at the edges of its tiles: a pass owns 48, 56 or 60 of its 64 columns by its rows
and precision, and runs levels in unrolled groups of 6 (prefetch 1) or 4 (prefetch 2).  Grids one column
either side of whole tiles, one row either side, and every remainder of the groups, against one step at a
time: the same bits."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from tests import decks
from tests.test_gpu_pairs import RX, TXS, COMPS

pytestmark = pytest.mark.gpu


def _run(precision, pairs, L, M, N, monkeypatch):
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    kw = dict(nx=L - 12, ny=M - 12, nz=N - 6)
    st = decks.small_setup(T, **kw)
    g = T.grid_arrays(st)
    cond = decks.layered_cond((N, M, L), g["Z"][:, None, None] * np.ones((1, M, L)), seed=4, blob=True)
    with T.Context(st, cond, precision) as c:
        assert (c.L, c.M, c.N) == (L, M, N)
        c.set_receivers(T.make_rxtime(0.02, 0.25, 8, 1, (1, 1, 1, 1, 1, 1)), RX)
        c.set_transmitters([T.make_tx(**TXS[0])])
        c.set_graph(0)
        c.set_pairs(*pairs)
        tr = c.run(0, 1, max_steps=150)[0]
        return tr, [c.get(q) for q in COMPS], c.pair_info()[2]


CASES = [(T.FP32, rows, pf, L, M, 20) for rows, pf, M in ((16, 1, 24), (16, 2, 25), (12, 1, 33), (14, 2, 31), (10, 1, 43))
         for L in (48, 49, 56, 57, 61, 97, 113)]
CASES += [(T.FP64, rows, pf, L, M, 20) for rows, pf, M in ((8, 1, 33), (11, 2, 36), (12, 1, 41)) for L in (56, 57, 113)]
CASES += [(p, 12, pf, 60, 32, N) for p in (T.FP32, T.FP64) for pf in (1, 2) for N in range(14, 21)]


@pytest.mark.parametrize("precision,rows,pf,L,M,N", CASES)
def test_pass_equals_single_steps(precision, rows, pf, L, M, N, monkeypatch):
    ref = _run(precision, (0, 1), L, M, N, monkeypatch)
    got = _run(precision, (rows, pf), L, M, N, monkeypatch)
    assert got[2] > 20 and ref[2] == 0
    assert np.abs(ref[0]).max() > 0 and np.array_equal(got[0], ref[0])
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b)
