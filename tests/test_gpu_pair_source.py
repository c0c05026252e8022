"""Source steps taken as pairs: the two-step pass patches a step's source cells (ElectricalFiled.cu:347-475) as it
passes their level, the cells above it are patched after each top launch.  Wires at each of the top levels (0: the
surface level; 1, 2, 3: either side of where the pass ends for the two steps), vertical and oblique wires over many
levels, wires of more cells than a wavefront has lanes and across tiles, several at once and none in a slot's tile:
the bits of one step at a time."""
import numpy as np
import pytest

import tcsem_fdtd_amd as T
from tests import decks, test_gpu_batch_pairs as B
from tests.test_gpu_pairs import COMPS, RX, _cond

pytestmark = pytest.mark.gpu

WIDE = dict(nx=130, ny=20, nz=14)
R4 = dict(rx_ids=[1, 2, 3, 4])
WIRES = {
    "level0": [dict(ort=1, bipolen=300.0, x=0.0, y=0.0, z=0.0, **R4)],
    "level1": [dict(ort=1, bipolen=300.0, x=0.0, y=0.0, z=50.0, **R4)],
    "level2": [dict(ort=2, bipolen=300.0, x=0.0, y=0.0, z=100.0, **R4)],
    "level3": [dict(ort=1, bipolen=300.0, x=0.0, y=0.0, z=150.0, **R4)],
    "vertical": [dict(ort=3, bipolen=600.0, x=0.0, y=0.0, z=300.0, **R4)],
    "oblique": [dict(ort=4, bipolen=500.0, x=0.0, y=0.0, z=250.0, azi=30.0, dip=40.0, **R4)],
    "long": [dict(ort=1, bipolen=4600.0, x=0.0, y=0.0, z=300.0, **R4)],
    "several": [dict(ort=1, bipolen=3000.0, x=500.0, y=0.0, z=200.0, **R4),
                dict(ort=3, bipolen=300.0, x=-1500.0, y=100.0, z=200.0, **R4),
                dict(ort=2, bipolen=400.0, x=1500.0, y=-100.0, z=100.0, **R4)],
}
SHAPES = [(T.FP32, 16, 2), (T.FP32, 10, 1), (T.FP64, 8, 2), (T.FP64, 11, 1)]


def _run(precision, pairs, wires, monkeypatch, steps=41):  # one step past the 40 of the wavelet
    monkeypatch.setenv("TCSEM_MARCH_ZCHUNKS", "1")
    with T.Context(decks.small_setup(T, **WIDE), _cond(WIDE), precision) as c:
        c.set_receivers(T.make_rxtime(0.02, 0.25, 16, 1, (1, 1, 1, 1, 1, 1)), RX)
        c.set_transmitters([T.make_tx(**t) for t in wires])
        c.set_graph(0)
        c.set_pairs(*pairs)
        c.run(0, len(wires), max_steps=steps)
        return [c.get(q, s) for s in range(len(wires)) for q in COMPS], c.pair_info()[2]


@pytest.mark.parametrize("precision,rows,pf", SHAPES)
@pytest.mark.parametrize("wires", sorted(WIRES))
def test_source_steps_in_pairs(precision, rows, pf, wires, monkeypatch):
    ref = _run(precision, (0, 1), WIRES[wires], monkeypatch)
    got = _run(precision, (rows, pf), WIRES[wires], monkeypatch)
    assert ref[1] == 0 and got[1] >= 18
    assert max(np.abs(f).max() for f in ref[0]) > 0
    for a, b in zip(got[0], ref[0]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("wire", ["level1", "level2", "vertical"])
@pytest.mark.parametrize("precision,rows", [(T.FP32, 16), (T.FP64, 11)])
def test_batch_source_steps_in_pairs(precision, rows, wire, monkeypatch):
    monkeypatch.setattr(B, "TX", WIRES[wire][0])
    tns = [0.25] * len(B.MODELS)
    ref = B._batch(precision, 0, tns, max_steps=40)
    got = B._batch(precision, rows, tns, max_steps=40)
    assert ref[3] == 0 and got[3] >= 18
    for key in ref[1]:
        assert np.array_equal(got[1][key], ref[1][key]), key
