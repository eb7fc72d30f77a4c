"""The closest hit over the tree is the closest hit over all triangles also where coordinates are small
against the ray's length, so that the rounding of a box's entry distance is larger than the box's padding:
the boxes of a tie must not be culled by it."""
import numpy as np
import pytest

from helpers import cull_scenes, twin_from_meshes


@pytest.mark.parametrize("name", ["chain", "flat"])
def test_closest_over_tree_is_closest_over_all(name):
    meshes, o, d = cull_scenes()[name]
    for builder in ("lbvh", "ploc"):
        tw = twin_from_meshes(meshes, builder=builder)
        t, prim = tw.brute_closest32(o, d)
        hits = tw.trace_closest(o, d)
        assert (prim >= 0).sum() > len(o) // 4
        np.testing.assert_array_equal(hits["prim"], prim)
        for tmax in (0.0, -1.0, -np.inf, np.nan):
            assert (tw.trace_closest(o[:200], d[:200], 0.0, tmax)["prim"] == -1).all()
