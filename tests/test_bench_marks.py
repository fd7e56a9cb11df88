"""bench.py's score-over-time marks: a trace that ended before the climb says
nothing about later times."""
import os
import sys

import numpy as np

from conftest import ROOT

sys.path.insert(0, ROOT)


def test_marks_of_whole_and_cut_traces():
    import bench

    tr, tt = np.array([10, 20, 30, 40]), np.array([1.0, 2.0, 3.0, 4.0])
    assert bench.score_marks(tr, tt, True, 5, 8.0, (0.25, 0.5, 1.0)) == {"2s": 20, "4s": 40, "8s": 40}
    assert bench.score_marks(tr, tt, False, 5, 8.0, (0.25, 0.5, 1.0)) == {"2s": 20, "4s": 40, "8s": None}
    none = np.zeros(0)
    assert bench.score_marks(none, none, True, 5, 8.0, (1.0,)) == {"8s": 5}
    assert bench.TRACE_CAP >= 60 * 20000
