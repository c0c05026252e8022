"""Two steps per pass need an intermediate state of five more fields.  Where the library takes pairs by itself and device
memory has no room for it (here: more is to stay free than the card has), runs and batches go on one step at a time,
with the same bits; where the caller asked for pairs they run."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from tests import decks

pytestmark = pytest.mark.gpu

RX = np.array([[150.0, 0.0, 400.0], [-200.0, -50.0, 350.0]])


@pytest.fixture(autouse=True)
def _unchunked(monkeypatch):
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", "fft")


def _ctx(precision, n=256):
    st = decks.small_setup(T, nx=n - 12, ny=n - 12, nz=16, pad=(2, 4))
    st.Az1 = st.Az2 = 0
    gi = T.grid_info(st)
    cond = decks.layered_cond((gi.N, gi.M, gi.L), T.grid_arrays(st)["Z"][:, None, None] * np.ones((1, gi.M, gi.L)),
                              seed=n)
    c = T.Context(st, cond, precision)
    c.set_receivers(T.make_rxtime(0.02, 0.25, 8, 1, (1, 1, 1, 1, 1, 1)), RX)
    c.set_transmitters([T.make_tx(1, 100.0, 0.0, 0.0, 300.0, [1, 2])])
    c.set_graph(0)
    return c


@pytest.mark.parametrize("precision", [T.FP64, T.FP32])
def test_run(precision, monkeypatch):
    with _ctx(precision) as c:
        ref = c.run(0, 1, max_steps=120)[0]
        assert c.pair_info()[2] > 40 and np.any(ref != 0)
    monkeypatch.setenv("TCSEM_SPARE_MB", "1e9")
    with _ctx(precision) as c:
        got = c.run(0, 1, max_steps=120)[0]
        assert c.pair_info()[0] == 0 and c.pair_info()[2] == 0
        assert np.array_equal(got, ref)
        c.set_pairs(8)
        assert np.array_equal(c.run(0, 1, max_steps=120)[0], ref)
        assert c.pair_info()[2] > 40


@pytest.mark.parametrize("precision", [T.FP64, T.FP32])
def test_batch(precision, monkeypatch):
    out = []
    for spare in ("0", "1e9"):
        monkeypatch.setenv("TCSEM_SPARE_MB", spare)
        cx = [_ctx(precision, n) for n in (256, 130)]
        try:
            with T.Batch(cx) as b:
                out.append(b.run(max_steps=120))
                rows, _, pairs = b.pair_info()
                assert (pairs > 40 and rows > 0) if spare == "0" else (pairs == 0 and rows == 0)
        finally:
            for c in cx:
                c.close()
    for a, g in zip(*out):
        assert np.any(a != 0) and np.array_equal(a, g)
