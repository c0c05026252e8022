"""bench.py prints HBM bytes beside a run only where the committed counters are of the shape that ran."""
import json
import os

import pytest

import bench

TABLE = json.load(open(os.path.join(bench.ROOT, "profiles", "traffic.json")))
ONE_STEP = {"rows": 10, "pf": 1, "zchunks": 2, "zsum": "fused", "sigma8": False, "pairs": None}


@pytest.mark.parametrize("key,res,entry", [
    ("large_5_fp32", {"pairs": {"rows": 16, "pf": 2}}, "large_5_fp32_pairs"),
    ("large_5_fp32", {"pairs": {"rows": 9, "pf": 2}}, None),
    ("large_5_fp64", {"pairs": {"rows": 11, "pf": 9}}, None),
    ("marine_3d_fp32", {"pairs": None, "tiling": ONE_STEP}, "marine_3d_fp32"),
    ("marine_3d_fp32", {"pairs": None, "tiling": dict(ONE_STEP, zchunks=1)}, None),
    ("marine_3d_fp32", {"pairs": None, "tiling": None}, None),
    ("uneven64_fp64", {"pairs": {"rows": 9}}, None)])
def test_only_the_shape_that_ran(key, res, entry):
    got = bench.counted_traffic(key, res)
    assert got == ((TABLE[entry]["bytes"], TABLE[entry]["tiling"]) if entry else (None, None))


def test_every_counted_shape_is_found():
    for key, v in TABLE.items():
        base, _, pairs = key.partition("_pairs")
        f = v["tiling"].split(",")
        if "_pairs" in key:
            res = {"pairs": {"rows": int(f[0]), "pf": int(f[1]) if len(f) > 1 else None}}
        elif len(f) == 2:
            res = {"pairs": None, "tiling": {"rows": int(f[0]), "pf": int(f[1])}}
        else:
            res = {"pairs": None, "tiling": {"rows": int(f[0]), "pf": int(f[1]), "zchunks": int(f[2]), "zsum": f[3],
                                             "sigma8": bool(int(f[4]))}}
        assert bench.counted_traffic(base, res) == (v["bytes"], v["tiling"]), key
