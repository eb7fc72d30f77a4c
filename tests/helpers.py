"""Shared helpers of the test suite: build the same scene on the GPU (product) and in the twin
(oracle), and compare."""
import math

import numpy as np


def twin_from_meshes(meshes, builder="lbvh"):
    import oracle
    from rendertoy_amd import scenes
    pos, nrm, uv, mo = scenes.triangle_arrays(meshes)
    has_n = [m.get("nrm") is not None for m in meshes]
    has_uv = [m.get("uv") is not None for m in meshes]
    return oracle.TwinScene(pos, nrm, uv, mo, has_n, has_uv, builder=builder)


def gpu_from_meshes(meshes, indexed=True):
    import rendertoy_amd as ren
    models = []
    for m in meshes:
        if indexed:
            mm = ren.mesh_from_arrays(m["pos"], m["idx"], m.get("nrm"), m.get("uv"))
        else:
            idx = m["idx"]
            mm = ren.mesh_from_arrays(m["pos"][idx].reshape(-1, 3), None,
                                      None if m.get("nrm") is None else m["nrm"][idx].reshape(-1, 3),
                                      None if m.get("uv") is None else m["uv"][idx].reshape(-1, 2))
        models.append(mm)
    return ren.Raycaster(models)


def gpu_arrays(rc):
    a = rc.scene_arrays()
    return {k: v.cpu().numpy() for k, v in a.items()}


def camera(eye=(0.0, 0.0, 3.0), target=(0.0, 0.0, 0.0), up=(0.0, 1.0, 0.0), fov=math.pi / 4,
           aspect=1.0):
    from rendertoy_amd._raycaster import Camera
    return Camera(eye, target, up, fov, aspect)


def random_rays(n, seed, box=1.5):
    """Rays from random origins on a sphere of radius 3 toward random points in the unit cube."""
    rng = np.random.default_rng(seed)
    o = rng.standard_normal((n, 3))
    o = 3.0 * o / np.linalg.norm(o, axis=1, keepdims=True)
    tgt = rng.uniform(-0.5 * box, 0.5 * box, (n, 3))
    d = tgt - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o.astype(np.float32), d.astype(np.float32)


def soa_tensors(o, d):
    import torch
    return {k: torch.from_numpy(np.ascontiguousarray(a[:, i])).cuda()
            for k, a, i in (("ox", o, 0), ("oy", o, 1), ("oz", o, 2),
                            ("dx", d, 0), ("dy", d, 1), ("dz", d, 2))}


def cull_scenes():
    """Scenes whose coordinates are small against their rays' length, with triangles that tie in t or
    almost: {name: (meshes, origins, directions)}."""
    rng = np.random.default_rng(11)

    def soup(tri):
        tri = np.asarray(tri, np.float32).reshape(-1, 3)
        return [{"pos": tri, "idx": np.arange(len(tri), dtype=np.int32).reshape(-1, 3), "nrm": None, "uv": None}]

    def aimed(k, distance, reach):
        o = rng.standard_normal((k, 3))
        o *= distance / np.linalg.norm(o, axis=1, keepdims=True)
        d = rng.uniform(-reach, reach, (k, 3)) - o
        return o.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)

    # triangles ever closer to x = 0, a seventh of them twice, along the axis
    x = 4.0 * np.float64(1.01) ** -np.arange(3000)
    z, s = np.zeros(3000), np.full(3000, 1e-3)
    one = np.stack([np.stack([x, z, z], 1), np.stack([x, s, z], 1), np.stack([x, z, s], 1)], 1)
    k = 5000
    o = np.stack([np.linspace(-1, 4.5, k), np.full(k, 2e-4), np.full(k, 2e-4)], 1).astype(np.float32)
    d = np.tile(np.float32([1, 0, 0]), (k, 1))
    d[1::2] *= -1
    out = {"chain": (soup(np.concatenate([one, one[::7]])), o, d)}
    # overlapping triangles in the plane z = 0, all of one t up to rounding
    f = rng.uniform(-1, 1, (700, 1, 3)) + rng.uniform(-0.3, 0.3, (700, 3, 3))
    f[..., 2] = 0.0
    out["flat"] = (soup(f), *aimed(4000, 3.0, 0.9))
    return out
