"""The three forms of the air boundary (line chain, tiled FFT chain, row operators), each forced through
TCSEM_UPCONT_CHAIN and confirmed by tcsem_air_form, on planes, runs, graph replays and model batches, whatever form
the library's own rule takes there.

Tolerances as the suite's others of the same comparison: planes 1e-12 (powers of two) and 1e-11 (Bluestein lengths,
in-place lines) in FP64, 2e-5 for FP32 transforms, 2e-6 for FP64 transforms of FP32 planes, 1e-6 for row operators in
FP32; traces 1e-9 (FP64) and 1e-4 (FP32) against the oracle; the same bits for graph replays and for FP64 batches of
unchunked marches."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from oracle import oracle as O
from tcsem_fdtd_amd import workloads as W
from tests import decks
from tests import test_gpu_batch as B

pytestmark = pytest.mark.gpu

FORM = {"lines": "lines", "fft": "fft", "dense": "matrix"}
BLUESTEIN = {"nx": 23, "ny": 17}
POW2 = {"nx": 72, "ny": 8, "pad": (2, 3), "arg": (1.5, 2.0)}      # 128 x 64
POW2_Y = {"nx": 10, "ny": 74, "pad": (3, 2), "arg": (1.3, 2.0)}   # 64 x 128
LONG_X = {"nx": 1100, "ny": 8, "pad": (2, 3), "arg": (1.5, 2.0)}  # L1 = 1156: working length 4096
LONG_Y = {"nx": 8, "ny": 550, "pad": (4, 3), "arg": (1.5, 2.9)}   # M1 above 1024 likewise
TALL = {"nx": 8, "ny": 804}                                       # more rows than the row operators take


def _plane(kw, precision, form, tol):
    so = decks.small_setup(O, **kw)
    m = O.Model(so)
    bz0 = np.random.default_rng(12).standard_normal((m.M, m.L))
    bxo, byo = m.upcont_plane(bz0)
    with T.Context(decks.small_setup(T, **kw), np.ones((m.N, m.M, m.L)), precision) as c:
        assert c.air_form()[0] == form
        bx, by = c.upcont_plane(bz0)
    assert decks.rel_l2(bx, bxo) < tol and decks.rel_l2(by, byo) < tol


@pytest.mark.parametrize("chain,precision,kw,tol", [
    ("fft", T.FP64, {}, 1e-12), ("fft", T.FP64, BLUESTEIN, 1e-11), ("fft", T.FP64, POW2, 1e-12),
    ("fft", T.FP64, POW2_Y, 1e-12), ("fft", T.FP32, {}, 2e-5), ("fft", T.FP32, BLUESTEIN, 2e-5),
    ("fft", T.FP32, POW2, 2e-5), ("fft", T.FP64, TALL, 1e-11), ("lines", T.FP64, LONG_X, 1e-11),
    ("lines", T.FP32, LONG_X, 2e-6), ("lines", T.FP64, LONG_Y, 1e-11), ("lines", T.FP64, TALL, 1e-11)])
def test_plane(chain, precision, kw, tol, monkeypatch):
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    _plane(kw, precision, FORM[chain], tol)


def test_plane_of_three_radix_passes(monkeypatch):
    """The 256 x 256 air plane of the 64 x 64 x 48 marine model on the tiled chain."""
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", "fft")
    d = W.marine_1d(T)
    m = O.Model(O.make_setup(**d.setup))
    assert (m.L1, m.M1) == (256, 256)
    bz0 = np.random.default_rng(4).standard_normal((m.M, m.L))
    bxo, byo = m.upcont_plane(bz0)
    with T.Context(T.make_setup(**d.setup), d.cond, T.FP64) as c:
        assert c.air_form()[0] == "fft"
        bx, by = c.upcont_plane(bz0)
    assert decks.rel_l2(bx, bxo) < 1e-12 and decks.rel_l2(by, byo) < 1e-12


@pytest.mark.parametrize("kw,form", [({}, "matrix"), (LONG_X, "matrix"), (TALL, "fft")])
def test_own_choice(kw, form):
    gi = T.grid_info(decks.small_setup(T, **kw))
    with T.Context(decks.small_setup(T, **kw), np.ones((gi.N, gi.M, gi.L)), T.FP64) as c:
        f, n = c.air_form()
        assert f == form and (n > 0) == (form == "matrix")


@pytest.mark.parametrize("precision", [T.FP32, T.FP64])
def test_own_choice_of_many_slots(precision):
    """Four slots share a read of the row operators: 32 slots of a shallow grid under 512 x 512 regular points read
    them eight times, which costs more than the transforms (778 us a step against 550 in FP32)."""
    st = decks.small_setup(T, nx=216, ny=216, nz=12, pad=(6, 14), arg=(1.05, 1.747))
    st.Az1 = st.Az2 = 0
    gi = T.grid_info(st)
    assert (gi.L, gi.M, gi.N, gi.L1, gi.M1) == (256, 256, 12, 512, 512)
    with T.Context(st, np.ones((gi.N, gi.M, gi.L)), precision) as c:
        assert [c.air_form(n)[0] for n in (16, 32)] == ["fft"] * 2


def test_operators_are_built_where_they_are_used(monkeypatch):
    """420 x 400 x 64 FP32: one transmitter stays with the chain, eight take the matrix form.  A context that never runs
    eight holds no operators, one that does runs them as a context that had them from the start, and its one-slot calls
    stay as they were."""
    st = decks.small_setup(T, nx=380, ny=360, nz=64, pad=(6, 14), arg=(1.05, 1.747))
    st.Az1 = st.Az2 = 0
    gi = T.grid_info(st)
    assert (gi.L, gi.M, gi.N) == (420, 400, 64)
    cond = np.ones((gi.N, gi.M, gi.L))
    bz0 = np.random.default_rng(5).standard_normal((gi.M, gi.L))
    txs = [T.make_tx(1, 100.0, 200.0 * q - 700.0, 0.0, 100.0, [1]) for q in range(8)]
    out = []
    for chain in ("", "dense"):
        monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
        with T.Context(st, cond, T.FP32) as c:
            c.set_receivers(B._rt(T), np.array([[0.0, 100.0, 400.0]]))
            c.set_transmitters(txs)
            if not chain:
                assert c.air_form(1) == ("fft", 0) and c.air_form(8)[0] == "matrix"
                plane = c.upcont_plane(bz0)
                c.begin(0, 1)
                assert c.air_form(1) == ("fft", 0)
            c.begin(0, 8)
            f, n = c.air_form(8)
            assert f == "matrix" and n > 2e8
            c.step(8)
            out.append([c.get(T.BXAIR, q) for q in range(8)])
            if not chain:
                assert c.air_form(1)[0] == "fft"
                for a, b in zip(plane, c.upcont_plane(bz0)):
                    assert np.array_equal(a, b)
    for a, b in zip(*out):
        assert np.any(a) and np.array_equal(a, b)


@pytest.mark.parametrize("precision,tol", [(T.FP64, 1e-11), (T.FP32, 2e-5)])
@pytest.mark.parametrize("chain", ["", "dense"])
@pytest.mark.parametrize("kw,form", [({}, "fft"), (BLUESTEIN, "fft"), (LONG_X, "lines"), (LONG_Y, "lines")])
def test_no_room_for_operators(kw, form, chain, precision, tol, monkeypatch):
    """Where device memory leaves no room for the row operators (here: more is to stay free than the card has), a
    context is created all the same and runs its FFT chain."""
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    monkeypatch.setenv("TCSEM_SPARE_MB", "1e9")
    _plane(kw, precision, form, tol)


TXS = [dict(B.TX, x=x, txid=q + 1) for q, x in enumerate((0.0, -100.0, 120.0, 60.0))]
COND = B.CONDS[0]
_REF = {}


def _oracle(q):
    if q not in _REF:
        m = O.Model(decks.small_setup(O), COND)
        _REF[q] = m.run(B._rt(O), B.RX, O.make_tx(**TXS[q]), max_steps=200)[0]
    return _REF[q]


def _context(precision, chain, kw={}, cond=COND):
    c = T.Context(decks.small_setup(T, **kw), cond, precision)
    assert c.air_form(4)[0] == FORM[chain]
    c.set_receivers(B._rt(T), B.RX)
    c.set_transmitters([T.make_tx(**t) for t in TXS])
    return c


@pytest.mark.parametrize("chain", ["lines", "fft", "dense"])
@pytest.mark.parametrize("precision,tol", [(T.FP64, 1e-9), (T.FP32, 1e-4)])
@pytest.mark.parametrize("ntx,pairs", [(1, 0), (1, 8), (3, 0), (3, 10)])
def test_run(chain, precision, tol, ntx, pairs, monkeypatch):
    """Single steps (the boundary beside the next march) and pairs (step A's boundary alone on the GPU)."""
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    with _context(precision, chain) as c:
        c.set_graph(0)
        c.set_pairs(pairs)
        got = c.run(0, ntx, max_steps=200)
        assert (c.pair_info()[2] > 0) == (pairs > 0)
    for q in range(ntx):
        assert np.all(decks.trace_error(got[q], _oracle(q)) < tol), q


@pytest.mark.parametrize("chain", ["lines", "fft", "dense"])
@pytest.mark.parametrize("ntx", [1, 3])
def test_graph_replays(chain, ntx, monkeypatch):
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    out = []
    for k in (0, 8):
        with _context(T.FP32, chain) as c:
            c.set_graph(k)
            out.append(c.run(0, ntx, max_steps=500))
            assert (c.graph_replays() > 3) == (k > 0)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_four_slots_at_the_most_rows(monkeypatch):
    """800 rows: four slots' columns of them take 154 KB of the 160 KB of LDS."""
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", "dense")
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    kw = {"nx": 8, "ny": 788, "nz": 4, "pad": (2, 4)}
    gi = T.grid_info(decks.small_setup(T, **kw))
    assert gi.M == 800
    cond = decks.layered_cond((gi.N, gi.M, gi.L), np.zeros((gi.N, gi.M, gi.L)), seed=6)
    with T.Context(decks.small_setup(T, **kw), cond, T.FP64) as c:
        c.set_receivers(B._rt(T), np.array([[50.0, 0.0, 100.0]]))
        c.set_transmitters([T.make_tx(1, 100.0, 0.0, 50.0 * q, 100.0, [1]) for q in range(4)])
        c.set_pairs(0)
        four = c.run(0, 4, max_steps=60)
        fields = [c.get(T.BXAIR, q) for q in range(4)]
        for q in range(4):
            assert np.array_equal(c.run(q, 1, max_steps=60)[0], four[q])
            assert np.any(fields[q]) and np.array_equal(c.get(T.BXAIR, 0), fields[q])


@pytest.mark.parametrize("chain", ["fft", "dense"])
@pytest.mark.parametrize("precision,tol", [(T.FP64, 0.0), (T.FP32, 1e-5)])
@pytest.mark.parametrize("rows", [0, 8])
def test_batch(chain, precision, tol, rows, monkeypatch):
    """Members equal the same models run alone."""
    monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    cx = [B._ctx(kw, cond, precision) for kw, cond in zip(B.MODELS, B.CONDS)]
    try:
        assert all(c.air_form()[0] == FORM[chain] for c in cx)
        alone = [c.run(0, 1, max_steps=300)[0] for c in cx]
        with T.Batch(cx) as b:
            b.set_pairs(rows)
            got = b.run(max_steps=300)
        for a, g in zip(alone, got):
            assert np.any(a != 0)
            assert np.array_equal(a, g) if tol == 0.0 else np.all(decks.trace_error(g, a) < tol)
    finally:
        for c in cx:
            c.close()


def _marine(n, nz):
    """A grid of n x n x nz cells under n + 256 regular points a side."""
    st = decks.small_setup(T, nx=n - 40, ny=n - 40, nz=nz, pad=(6, 14), arg=(1.05, 1.747))
    st.Az1 = st.Az2 = 0
    return st


@pytest.mark.parametrize("precision,tol", [(T.FP64, 1e-11), (T.FP32, 1e-5)])
@pytest.mark.parametrize("rows", [0, 8])
@pytest.mark.parametrize("sides,form", [((256, 100, 100), "matrix"), ((256, 256, 100), "fft")])
def test_batch_form(sides, form, precision, tol, rows):
    """The batch's members together decide: a 256 x 256 grid alone stays with the chain, and two of 100 x 100 carry it
    over to row operators built for the batch, unless a second one of 256 x 256 comes with it.  Each member equals its
    run alone to round-off."""
    cx = []
    try:
        for q, n in enumerate(sides):
            st = _marine(n, 24)
            gi = T.grid_info(st)
            cond = decks.layered_cond((gi.N, gi.M, gi.L), T.grid_arrays(st)["Z"][:, None, None] *
                                      np.ones((1, gi.M, gi.L)), seed=q)
            c = T.Context(st, cond, precision)
            c.set_receivers(B._rt(T, 0.08 if q == 1 else 0.25), B.RX)
            c.set_transmitters([T.make_tx(**B.TX)])
            c.set_pairs(8)
            c.set_graph(0)
            cx.append(c)
            assert c.air_form()[0] == ("fft" if n == 256 else "matrix")
        alone = [c.run(0, 1, max_steps=300)[0] for c in cx]
        with T.Batch(cx) as b:
            b.set_pairs(rows)
            b.enable_timing()
            assert b.air_form() == form
            got = b.run(max_steps=300)
            assert b.timing()["upcont_ms"] > 0.0
        for c, n, a, g in zip(cx, sides, alone, got):
            assert np.any(a != 0)
            assert np.all(decks.trace_error(g, a) < tol)
        again = [c.run(0, 1, max_steps=300)[0] for c in cx]  # a member keeps its own form, operators or not
        for a, g in zip(alone, again):
            assert np.array_equal(a, g)
    finally:
        for c in cx:
            c.close()


def test_batch_without_room_for_a_member_s_operators(monkeypatch):
    cx = []
    try:
        for q, n in enumerate((256, 100, 100)):  # a batch in matrix form, above
            st = _marine(n, 24)
            gi = T.grid_info(st)
            cx.append(T.Context(st, np.ones((gi.N, gi.M, gi.L)), T.FP64))
            cx[-1].set_receivers(B._rt(T), B.RX)
            cx[-1].set_transmitters([T.make_tx(**B.TX)])
            cx[-1].set_pairs(8)
        alone = [c.run(0, 1, max_steps=100)[0] for c in cx]
        monkeypatch.setenv("TCSEM_SPARE_MB", "1e9")
        with T.Batch(cx) as b:
            assert b.air_form() == "fft"
            got = b.run(max_steps=100)
        for a, g in zip(alone, got):
            assert np.all(decks.trace_error(g, a) < 1e-11)
    finally:
        for c in cx:
            c.close()


def test_batch_of_a_member_without_the_matrix_form(monkeypatch):
    cx = []
    try:
        for kw, cond, chain in zip(B.MODELS, B.CONDS, ("dense", "fft")):
            monkeypatch.setenv("TCSEM_UPCONT_CHAIN", chain)
            cx.append(B._ctx(kw, cond, T.FP64))
        with T.Batch(cx) as b:
            assert b.air_form() == "fft"
            b.run(max_steps=60)
    finally:
        for c in cx:
            c.close()
