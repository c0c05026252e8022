"""The air boundary in matrix form (row operators per x wavenumber) against the FP64 oracle, forced on
and off where the library would choose the other: plane sizes either side of the kernels' 16- and
32-wide tiles, odd and even irregular and regular sides (the y-Nyquist bin, a middle row), stretched
cells (dx != dy), several slots.

FP64: sums of up to M1 products of rounded tables, at most a few thousand round-offs of 1.1e-16, and the
oracle's own transforms: 1e-11, as the FFT chains' Bluestein planes.  FP32 contexts keep the plane and the row operators in FP32 (6e-8 each) and sum in
FP64: 1e-6."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from oracle import oracle as O
from tests import decks

pytestmark = pytest.mark.gpu

# nx, ny, pad, growth: L = nx + 2 (outer + inner)
PLANES = {
    "18x18": {"nx": 6, "ny": 6},
    "32x31": {"nx": 20, "ny": 19},
    "33x32": {"nx": 21, "ny": 20},
    "64x65_wide": {"nx": 36, "ny": 37, "pad": (6, 8), "arg": (1.05, 1.6)},
    "128x64_pow2": {"nx": 72, "ny": 8, "pad": (2, 3), "arg": (1.5, 2.0)},
    "97x130": {"nx": 85, "ny": 118},
}


def _check(kw, precision, tol, dy=None):
    so, st = decks.small_setup(O, **kw), decks.small_setup(T, **kw)
    if dy:
        so.dymin = st.dymin = dy
    m = O.Model(so)
    bz0 = np.random.default_rng(11).standard_normal((m.M, m.L))
    bxo, byo = m.upcont_plane(bz0)
    with T.Context(st, np.ones((m.N, m.M, m.L)), precision) as c:
        bx, by = c.upcont_plane(bz0)
    assert decks.rel_l2(bx, bxo) < tol and decks.rel_l2(by, byo) < tol
    return m


@pytest.mark.parametrize("chain", ["dense", "fft"])
@pytest.mark.parametrize("precision", [T.FP64, T.FP32])
@pytest.mark.parametrize("name", sorted(PLANES))
def test_plane(name, precision, chain, monkeypatch):
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    tol = 1e-11 if precision == T.FP64 else (1e-6 if chain == "dense" else 2e-5)
    _check(PLANES[name], precision, tol)


def test_plane_of_unequal_cells(monkeypatch):
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", "dense")
    _check({"nx": 23, "ny": 17}, T.FP64, 1e-11, dy=40.0)


def test_plane_beyond_the_tiled_chain():
    """M1 = 1156 (working length 4096 along y): the matrix form without being asked for."""
    m = _check({"nx": 8, "ny": 1100 // 2, "pad": (4, 3), "arg": (1.5, 2.9)}, T.FP64, 1e-11)
    assert m.M1 > 1024


@pytest.mark.parametrize("precision", [T.FP64, T.FP32])
def test_slots_equal_single_runs(precision, monkeypatch):
    """1, 2, 3 and 5 slots (one, two and four share a read of the row operators): the same bits."""
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")  # the march's own choice depends on the slots
    st = decks.small_setup(T)
    gi, g = T.grid_info(st), T.grid_arrays(st)
    cond = decks.layered_cond((gi.N, gi.M, gi.L), g["Z"][:, None, None] * np.ones((1, gi.M, gi.L)), seed=3)
    rx = np.array([[150.0, 0.0, 400.0], [300.0, 50.0, 400.0]])
    out = []
    with T.Context(st, cond, precision) as c:
        c.set_receivers(T.make_rxtime(0.02, 0.2, 8, 1, (1, 1, 1, 1, 1, 1)), rx)
        c.set_transmitters([T.make_tx(1, 100.0, 40.0 * q - 80.0, 0.0, 300.0, [1, 2]) for q in range(5)])
        for n in (5, 3, 2, 1):
            out.append(c.run(0, n, max_steps=120))
    for o in out[1:]:
        for b, t in enumerate(o):
            assert np.array_equal(t, out[0][b]), (len(o), b)
