"""The stacks of the walks that take several entries a step hold what the deepest, widest tree can push: past a
switch they go on one entry at a time, and end within their share of LDS."""
import os
import re

import pytest

from helpers import deep_wide_scene, group_walk_peak, twin_from_meshes

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rendertoy_amd", "csrc",
                   "rt_trace_shared.h")


@pytest.mark.parametrize("lanes", [16, 64])
def test_peak_past_the_switch(lanes):
    words = int(re.search(r"constexpr int kGroupWords = (\d+);", open(SRC).read()).group(1))
    assert "kSwitch = kCap - 3 * E - 93" in open(SRC).read()
    peak, single, switch, cap = group_walk_peak(twin_from_meshes(deep_wide_scene()).nodes4, lanes, words)
    assert switch < peak <= cap and single > 20
