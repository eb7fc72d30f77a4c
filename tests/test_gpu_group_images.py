"""Camera and render of images small enough that 16 or 64 lanes take each pixel, against the twin bit
for bit: sizes on both sides of every switch and partial 8x8 blocks, with and without counts."""
import numpy as np
import pytest
import torch

from helpers import camera, gpu_from_meshes, twin_from_meshes

pytestmark = pytest.mark.gpu

LIGHT = (np.array([1.0, 1.0, 1.0], np.float32) / np.float32(np.sqrt(3.0))).astype(np.float32)


def _u32(a):
    return np.ascontiguousarray(a).view(np.uint32)


# 722 triangles: 64 lanes to 4,096 pixels, 16 to 24,182; 28,802: 64 lanes to 4,800 pixels
@pytest.mark.parametrize("freq,sizes", [(6, ((1, 1), (3, 5), (9, 17), (64, 64), (17, 241), (155, 156), (157, 155))),
                                        (38, ((75, 64), (4801, 1)))])
def test_group_images(ren, freq, sizes):
    from rendertoy_amd import scenes
    meshes = [scenes.icosphere(freq, 41), scenes.ground_plane()]
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    tex = scenes.value_noise_rgba8(32, 42)
    for w, h in sizes:
        cam = camera(eye=(0.8, 0.5, 1.9), aspect=w / h)
        ref = tw.trace_camera(cam.as_array(), w, h)
        hits = rc.cast_camera(cam, w, h)
        for k in ("t", "u", "v", "prim"):
            np.testing.assert_array_equal(_u32(hits[k].cpu().numpy()), _u32(ref[k]))
        args = dict(light=LIGHT, textures=[torch.from_numpy(tex).cuda()], mesh_textures=[0, -1])
        rgb, t, prim, st = tw.render(cam.as_array(), w, h, LIGHT, textures=[tex], mesh_tex=[0, -1])
        stats = torch.zeros(4, dtype=torch.int32, device="cuda")
        for s in (None, stats):
            img, out = rc.render(cam, w, h, return_hits=True, stats=s, **args)
            np.testing.assert_array_equal(_u32(img.cpu().numpy()), _u32(rgb))
            np.testing.assert_array_equal(out["prim"].cpu().numpy(), prim)
            np.testing.assert_array_equal(_u32(out["t"].cpu().numpy()), _u32(t))
        assert list(stats.cpu().numpy()[:3]) == list(st)
