"""Path frames on either side of the sizes at which groups of lanes walk their rays: the radiance and ray
counts of the per-lane traversals, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import gpu_from_meshes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(ren):
    from rendertoy_amd import scenes
    return gpu_from_meshes([scenes.icosphere(24, 5), scenes.ground_plane()])


@pytest.mark.parametrize("bounces", [0, 2])
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (7, 5, 3), (64, 64, 1), (241, 17, 1), (128, 256, 1), (99, 331, 1),
                                     (61, 37, 17), (362, 362, 1), (363, 362, 1)])
def test_groups_match_lanes(ren, scene, w, h, spp, bounces):
    cam = ren.Camera((0.4, 0.9, 1.6), (0.0, -0.2, 0.0), aspect=w / h)

    def frame(tuning):
        counts = torch.zeros(bounces + 1, dtype=torch.int32, device="cuda")
        out = scene.trace_paths(cam, w, h, spp=spp, bounces=bounces, seed=9, counts=counts, tuning=tuning)
        return out.cpu().numpy().view(np.uint32), counts.cpu().numpy()
    image, counts = frame(None)
    from rendertoy_amd import _native
    want, want_counts = frame({"primary": "lane", "lane_stack": _native.RT_LANE_STACK_MAX - 1})
    np.testing.assert_array_equal(image, want)
    np.testing.assert_array_equal(counts, want_counts)
