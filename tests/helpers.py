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


def deep_wide_scene():
    """Meshes whose 4-wide tree is a spine of full nodes, each sibling with 16 inner grandchildren, every box of
    which holds the unit cube: a ray from inside enters them all and walks that take several entries of their
    stack a step pile the siblings up. One triangle in the plane x - y = const per Morton code, several per
    code at the siblings' leaves."""
    rng = np.random.default_rng(7)
    codes = []
    for level in range(15):  # 2 bits of the 30 per 4-wide level; the spine is 11 11 11 ...
        spine = ((1 << (2 * level)) - 1) << (30 - 2 * level)
        for sib in range(3):
            base = spine | sib << (28 - 2 * level)
            free = 28 - 2 * level  # bits below the sibling's
            for k in range(16):
                code = base | (k << (free - 4) if free >= 4 else k >> (4 - free))
                codes += [code] * 8
    codes += [(1 << 30) - 1] * 40960  # the spine's end: codes alike, split by slot
    codes = np.array(sorted(codes), np.int64)

    def compact(c):  # every third bit
        return sum(((c >> np.int64(3 * b)) & 1) << np.int64(b) for b in range(10))
    q = np.stack([compact(codes >> 2), compact(codes >> 1), compact(codes)], 1)
    centre = (q + 0.5) / 1024.0
    tri = centre[:, None, :] + 4.0 * np.array([[-1, -1, -1], [1, 1, 1], [1, 1, -1]])[None]
    pos = tri[rng.permutation(len(tri))].reshape(-1, 3).astype(np.float32)
    idx = np.arange(len(pos), dtype=np.int32).reshape(-1, 3)
    return [{"pos": pos, "idx": idx, "nrm": None, "uv": None}]


def group_walk_peak(nodes4, lanes, words=1024):
    """(highest number of stack entries, steps of one entry) of a walk of `lanes` lanes per ray that enters every
    box, by the rules of the device's group_walk."""
    entries, cap = lanes // 4, words * lanes // 64
    switch = cap - 3 * entries - 93
    refs = np.asarray(nodes4, np.float32).reshape(-1, 32)[:, 24:28].copy().view(np.int32)
    stack, peak, single = [0], 1, 0
    while stack:
        k = 1 if len(stack) > switch else min(len(stack), entries)
        single += len(stack) > switch
        taken, stack = stack[-k:], stack[:-k]
        for node in taken:
            stack += [int(r) for r in refs[node] if 0 <= r < 0x7FFFFFFF]
        peak = max(peak, len(stack))
        assert peak <= cap, "a group's stack would run into its neighbour's"
    return peak, single, switch, cap
