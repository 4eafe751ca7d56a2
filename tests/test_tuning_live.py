"""Which launch shapes act on which class, and that the tuner times each launch
once and picks no shape that launches the same as the default (host side)."""
import os

import numpy as np
import pytest

from aeroapps_amd import tune as T
from aeroapps_amd._lib import LIB_PATH

pytestmark = pytest.mark.skipif(not os.path.exists(LIB_PATH), reason="library not built")


def test_live_shapes_per_class():
    # n <= 15 in FP64 and n <= 7 mixed have no band solver; FP64 has no SAB/DAB kernel there
    assert T.live(6, 1, 0) == (False, False) and T.live(2, 3, 0) == (False, False)
    assert T.live(6, 1, 1) == (False, True) and T.live(2, 1, 1) == (False, True)
    assert T.live(8, 1, 0) == (False, False) and T.live(8, 1, 1) == (True, True)
    # one shape only
    assert T.live(12, 1, 1) == (False, False) and T.live(16, 1, 0) == (False, False)
    assert T.live(2, 3, 1) == (False, False)


@pytest.mark.parametrize("N,precision,launches", [(6, 0, 1), (6, 1, 2), (8, 0, 1), (8, 1, 4)])
def test_tuner_times_each_launch_once(monkeypatch, N, precision, launches):
    shapes = []

    class Stub:
        def __init__(self, torch, ncol, nstreams, nstokes):
            pass

        def run(self, prec):
            t = T.get_tuning(N, 1, prec)
            shapes.append((t["bvp_lanes"], t["sab_pairs"]))
            return 1.0 / len(shapes)   # whatever comes later is faster

        def outputs(self):
            return np.zeros(1), np.zeros(1, dtype=np.int32)

        def close(self):
            pass

    monkeypatch.setattr(T, "Sample", Stub)
    try:
        best, times = T.tune_class(None, N, 1, (precision,), ncol=1, reps=1, log=lambda m: None)[precision]
        assert len(set(shapes)) == launches
        assert sorted(times) == T.shape_candidates(N, 1)
        default = T.get_tuning(N, 1, precision)
        bvp, sab = T.live(N, 1, precision)
        assert bvp or best[0] == default["bvp_lanes"]
        assert sab or best[1] == default["sab_pairs"]
    finally:
        T.load_tuning(None)
