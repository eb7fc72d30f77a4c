"""Ray buffers small enough that 16 or 64 lanes walk each ray, against the twin bit for bit: sizes on
both sides of every switch (rays per wave, lanes per ray, one-lane walks), a root that is a leaf, an
empty scene, per-ray intervals and deep chains."""
import numpy as np
import pytest

from helpers import gpu_from_meshes, random_rays, soa_tensors, twin_from_meshes

pytestmark = pytest.mark.gpu


def _u32(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _check(rc, tw, o, d, tmin=0.0, tmax=np.inf):
    rays = soa_tensors(o, d)
    ref = tw.trace_closest(o, d, tmin, tmax)
    hits = rc.trace_soa(rays, tmin=tmin, tmax=tmax)
    np.testing.assert_array_equal(hits["prim"].cpu().numpy(), ref["prim"])
    for k in ("t", "u", "v"):
        np.testing.assert_array_equal(_u32(hits[k].cpu().numpy()), _u32(ref[k]))
    np.testing.assert_array_equal(rc.occluded(rays, tmin=tmin, tmax=tmax).cpu().numpy(), tw.trace_any(o, d, tmin, tmax))


@pytest.mark.parametrize("freq,sizes", [(6, (1, 3, 4, 5, 63, 4096, 4097, 65536, 65537)), (60, (1, 2, 9000, 9001)),
                                        (112, (31361, 131072, 131073))])
def test_group_walk_sizes(ren, freq, sizes):
    from rendertoy_amd import scenes
    meshes = [scenes.icosphere(freq, 31), scenes.ground_plane()]
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    o, d = random_rays(max(sizes), 5)
    o[::2] *= np.float32(0.15)  # half of the rays start inside
    for n in sizes:
        _check(rc, tw, o[:n], d[:n])
        _check(rc, tw, o[:n], d[:n], 0.3, 1.7)


@pytest.mark.parametrize("tris", [0, 1, 4, 5])
def test_group_walk_tiny_scenes(ren, tris):
    rng = np.random.default_rng(tris)
    pos = rng.uniform(-0.5, 0.5, (3 * tris, 3)).astype(np.float32)
    meshes = [{"pos": pos, "idx": np.arange(3 * tris, dtype=np.int32).reshape(-1, 3), "nrm": None, "uv": None}]
    rc = gpu_from_meshes(meshes)
    o, d = random_rays(5000, 7)
    if tris == 0:
        for n in (7, 5000):
            assert (rc.trace_soa(soa_tensors(o[:n], d[:n]))["prim"] == -1).all()
            assert not rc.occluded(soa_tensors(o[:n], d[:n])).any()
        return
    tw = twin_from_meshes(meshes)
    for n in (7, 5000):
        _check(rc, tw, o[:n], d[:n])


def test_group_walk_long_stacks(ren):
    """Rays along a chain of thousands of nested boxes enter every child they meet, and the triangles
    near the chain's end tie in t: stacks grow past the depth-first switch and the smaller primitive
    wins, as over all triangles."""
    x = 4.0 * np.float64(1.01) ** -np.arange(3000)
    z, s = np.zeros(3000), np.full(3000, 1e-3)
    one = np.stack([np.stack([x, z, z], 1), np.stack([x, s, z], 1), np.stack([x, z, s], 1)], 1).astype(np.float32)
    tri = np.concatenate([one, one[::7]]).reshape(-1, 3)
    meshes = [{"pos": tri, "idx": np.arange(len(tri), dtype=np.int32).reshape(-1, 3), "nrm": None, "uv": None}]
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    k = 5000
    o = np.stack([np.linspace(-1, 4.5, k), np.full(k, 2e-4), np.full(k, 2e-4)], 1).astype(np.float32)
    d = np.tile(np.float32([1, 0, 0]), (k, 1))
    d[1::2] *= -1
    t, prim = tw.brute_closest32(o, d)
    for n in (200, k):
        hits = rc.trace_soa(soa_tensors(o[:n], d[:n]))
        np.testing.assert_array_equal(hits["prim"].cpu().numpy(), prim[:n])
        np.testing.assert_array_equal(rc.occluded(soa_tensors(o[:n], d[:n])).cpu().numpy(), prim[:n] >= 0)
