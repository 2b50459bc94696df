"""bench.py's rates of the motion producer's full-size level, from profile
steps as kvpersist.motion.farneback_profile returns them."""

import sys
from pathlib import Path

import pytest

from kvpersist import motion

sys.path.insert(0, str(Path(__file__).resolve().parent.parent))
import bench  # noqa: E402

BLUR, EXPAND, INIT, FLOW = motion.KINDS[1:5]


def _steps(merged):
    flows = [(FLOW, lv, 1.0) for lv in (3, 2, 1)]
    head = [(BLUR, 1, 2.0), (EXPAND, 0 if merged else 1, 3.0)]
    return head + flows + [(EXPAND, 0, 0.5)] * (not merged) + [(INIT, 0, 0.25), (FLOW, 0, 1.0),
                                                               (FLOW, 0, 2.0)]


@pytest.mark.parametrize("merged", [True, False])
def test_only_passes_of_the_full_size_level_alone_are_rated(merged):
    """Short clips expand all levels in one step, labelled 0: it has no level-0 rate."""
    roofs = bench.motion_level0(_steps(merged), 10, 1000)
    assert set(roofs) == {INIT, FLOW} | (set() if merged else {EXPAND})
    flow = roofs[FLOW]
    assert flow["passes_per_clip"] == 2 and flow["avg_pass_ms"] == 1.5
    assert flow["bytes_per_pass"] == bench.MOTION_BYTES_PER_PX[FLOW] * 1000 * 9
    if not merged:
        assert roofs[EXPAND]["bytes_per_pass"] == bench.MOTION_BYTES_PER_PX[EXPAND] * 1000 * 10


def test_one_level_is_rated_alone():
    roofs = bench.motion_level0([(EXPAND, 0, 1.0), (FLOW, 0, 1.0)], 2, 1000)
    assert set(roofs) == {EXPAND, FLOW}


def test_kind_names_are_those_of_the_launches_that_exist():
    assert motion.KINDS == ("", "preblur", "poly_exp", "init_flow", "flow", "matrices")
    assert set(bench.MOTION_BYTES_PER_PX) < set(motion.KINDS)
