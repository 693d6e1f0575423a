"""The benchmark's one result line stays short: a reader that keeps the last
kilobytes of the output must find it whole."""
import json
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("runs", [2, 60, 500])
def test_guiding_statistics_do_not_grow_with_the_runs(runs):
    """Five regions of these are the longest part of the line."""
    rng = np.random.default_rng(runs)
    g, p, c = rng.lognormal(0.0, 2.0, (3, runs))
    side = bench.guide_side(g, p, c)
    assert len(json.dumps(side)) < 900
    assert side["relmse_ratio_equal_time"] == pytest.approx(g.mean() / p.mean())
    assert side["common_seeds"]["runs_guided_below_plain"] == int((g < c).sum())
    lo, hi = side["common_seeds"]["relmse_ratio_ci95"]
    assert lo <= hi
