"""bench.py's account of a run's launches: every step is in one, the last one is
a single step, and captured graphs hold whole launches."""
import pytest

import bench


@pytest.mark.parametrize("form, per", [("single", 1), ("pair", 2), ("march", 7), ("march", 4),
                                       ("tile", 8), ("tile", 4)])
def test_launches_cover_the_steps(form, per):
    for steps in list(range(1, 300)) + [1000, 2000]:
        multi, single, graphed = bench.launch_plan(form, per, steps)
        assert single >= 1 and graphed <= steps and graphed % per == 0
        if form == "tile":  # a rest of two steps and more is a launch of its own
            assert per * (multi - 1) + 2 <= steps - single <= per * multi or multi == 0
            assert single <= 2
        else:
            assert per * multi * (per > 1) + single == steps
            assert single <= per or per == 1


def test_headline_runs():
    assert bench.launch_plan("pair", 2, 20) == (9, 2, 0)
    assert bench.launch_plan("pair", 2, 2000) == (999, 2, 1984)
