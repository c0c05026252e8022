"""bench.py's timed window holds the same steps of the run whether or not the model is timed one step at a time first:
its FP32 and FP64 fields are compared after it."""
import numpy as np
import pytest

import bench
import tcsem_fdtd_amd as T
from tcsem_fdtd_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_one_step_timing_leaves_the_window(monkeypatch):
    monkeypatch.setenv("TCSEM_MARCH_PAIRS", "8,1")
    deck = W.marine_1d(T)
    a = bench.gpu_run(T, deck, T.FP64, 1, 12, 4, tune=False)
    b = bench.gpu_run(T, deck, T.FP64, 1, 12, 4, tune=False, one_step_too=True)
    assert a["one_step"] is None and b["one_step"]["value"] > 0
    assert np.any(a["ex"] != 0) and np.linalg.norm(b["ex"] - a["ex"]) < 1e-10 * np.linalg.norm(a["ex"])
