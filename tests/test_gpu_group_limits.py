"""Where groups of lanes take over from the one-lane and packet walks: the same results on both sides of every
size, and no longer time past it than the walk they replace where all rays' walks are alike."""
import math

import numpy as np
import pytest
import torch

from helpers import camera, gpu_from_meshes, random_rays, soa_tensors, twin_from_meshes

pytestmark = pytest.mark.gpu


def _u32(a):
    return np.ascontiguousarray(a).view(np.uint32)


# 722 triangles: 64 lanes to 4,096 rays, images to 24,183 pixels; 317,522: 52,920 pixels and 39,690 rays, 379,807
@pytest.mark.parametrize("freq,images,rays", [
    (6, ((64, 64), (4097, 1), (155, 156), (24184, 1)), (4096, 4097, 65536, 65537)),
    (126, ((210, 252), (52921, 1), (612, 620), (613, 620)), (39690, 39691, 65536, 65537, 131072, 131073))])
def test_same_hits_on_both_sides(ren, freq, images, rays):
    from rendertoy_amd import scenes
    meshes = [scenes.icosphere(freq, 17), scenes.ground_plane()]
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    for w, h in images:
        cam = camera(eye=(0.8, 0.5, 1.9), aspect=w / h)
        ref, hits = tw.trace_camera(cam.as_array(), w, h), rc.cast_camera(cam, w, h)
        for k in ("t", "u", "v", "prim"):
            np.testing.assert_array_equal(_u32(hits[k].cpu().numpy()), _u32(ref[k]))
    o, d = random_rays(max(rays), 5)
    o[::2] *= np.float32(0.15)  # half of the rays start inside
    for n in rays:
        soa = soa_tensors(o[:n], d[:n])
        ref, hits = tw.trace_closest(o[:n], d[:n]), rc.trace_soa(soa)
        for k in ("t", "u", "v", "prim"):
            np.testing.assert_array_equal(_u32(hits[k].cpu().numpy()), _u32(ref[k]))
        np.testing.assert_array_equal(rc.occluded(soa).cpu().numpy(), tw.trace_any(o[:n], d[:n]))


@pytest.mark.parametrize("freq,frames", [
    (6, ((64, 64), (4097, 1), (128, 256), (32769, 1), (362, 362), (363, 362))),
    (126, ((128, 128), (16385, 1), (256, 256), (65537, 1), (512, 512), (513, 512)))])
def test_same_paths_on_both_sides(ren, freq, frames):
    from rendertoy_amd import scenes
    rc = gpu_from_meshes([scenes.icosphere(freq, 17), scenes.ground_plane()])
    for w, h in frames:
        cam = ren.Camera((0.4, 0.9, 1.6), (0.0, -0.2, 0.0), aspect=w / h)
        images = [rc.trace_paths(cam, w, h, spp=1, bounces=2, seed=9, tuning=t)
                  for t in (None, {"primary": "lane", "lane_stack": 31})]
        assert torch.equal(images[0], images[1])


def _time(f):
    f()
    times = []
    for _ in range(11):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(200000)  # the launches queue up behind it
        a.record()
        f()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


@pytest.fixture(scope="module")
def near_view(ren):
    """A sphere seen from so near that all rays hit and their walks are alike; a room around the origin."""
    from rendertoy_amd import scenes
    out = []
    for freq, scale in ((126, 1.0), (63, 4.0)):
        m = dict(scenes.icosphere(freq, 3))
        m["pos"] = m["pos"] * np.float32(scale)
        out.append(gpu_from_meshes([m]))
    return out


@pytest.mark.parametrize("w,h", [(640, 620), (768, 512)])
def test_time_of_images(ren, near_view, w, h):
    cam = ren.Camera((0.1, 0.2, 0.8), (0, 0, 0), (0, 1, 0), math.pi / 4, w / h)
    for rc in near_view:
        took = _time(lambda: rc.cast_camera(cam, w, h))
        packets = _time(lambda: rc.cast_camera(cam, w, h, tuning={"super_tile": 1}))
        assert took < 1.4 * packets, (took, packets)


@pytest.mark.parametrize("n", [100000, 131072])
def test_time_of_rays(ren, near_view, n):
    side = int(math.sqrt(n))
    cam = ren.Camera((0.1, 0.2, 0.8), (0, 0, 0), (0, 1, 0), math.pi / 4, 1.0)
    coherent = {k: v.clone() for k, v in near_view[0].generate_rays(cam, side, side).items()}
    for rc in near_view:
        for rays in (coherent, soa_tensors(*random_rays(n, 2))):
            took, lanes = _time(lambda: rc.trace_soa(rays)), _time(lambda: rc.trace_soa(rays, tuning={"lane_stack": 31}))
            assert took < 1.3 * lanes, (took, lanes)
