"""Path frames at every number of samples the camera kernel's waves split differently (one wave each
for up to 4 at a time), on partial 8x8 blocks, against the twin bit for bit."""
import numpy as np
import pytest
import torch

from helpers import camera, gpu_from_meshes, twin_from_meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spp", [1, 2, 3, 4, 5, 9])
def test_samples(ren, spp):
    from rendertoy_amd import scenes
    meshes = [scenes.icosphere(7, 61), scenes.ground_plane()]
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    for w, h, bounces in ((37, 21, 2), (1, 3, 1), (8, 8, 0)):
        cam = camera(eye=(0.3, 0.9, 1.8), aspect=w / h)
        counts = torch.zeros(bounces + 1, dtype=torch.int32, device="cuda")
        img = rc.trace_paths(cam, w, h, spp=spp, bounces=bounces, seed=9, frame=spp, counts=counts)
        rad, _, cnt = tw.paths(cam.as_array(), w, h, spp=spp, bounces=bounces, seed=9, frame=spp)
        np.testing.assert_array_equal(img.cpu().numpy().reshape(-1).view(np.uint32), rad.view(np.uint32))
        assert list(counts.cpu().numpy()) == list(cnt)
