"""Performance cases of the ray caster: the calls a user's program makes, over the sizes it makes them at.

Scenes are displaced geodesic spheres of 500 to 1.3 million triangles, mostly on a ground plane, as
in the benchmark and the tests; a case's seed moves every vertex, ray, eye and texel. The kinds:

  build     Raycaster(meshes): the hierarchy of a scene that was loaded or has moved; run() returns
            every array of the built scene
  camera    Raycaster.cast_camera: closest hits of an image's primary rays
  cast      Raycaster.ray_cast: closest hits of a Ray buffer (picking, lidar, probes)
  segments  Raycaster.occluded: visibility between pairs of points, SoA rays with their own tmax
  render    Raycaster.render: shaded, textured, shadowed image
  batch     BatchRender.launch: many small images of several scenes at once
  paths     Raycaster.trace_paths: diffuse light, several samples and bounces
  normals   compute_normals: vertex normals of an imported or deformed mesh
"""
import functools
import math

import numpy as np
import torch

import rendertoy_amd as ren
from rendertoy_amd import scenes
from rendertoy_amd._raycaster import TextureBinding
from rendertoy_amd.batch import BatchRender, RenderRequest

LIGHT = np.ones(3) / math.sqrt(3.0)


def listed():
    return [
        # a preview or thumbnail: one small image, nothing to hide the call's latency behind
        {"name": "render thumbnail", "kind": "render", "freq": 8, "width": 128, "height": 128,
         "texture": 64, "bilinear": True, "shadows": True},
        # a pick under the mouse, a handful of probe rays
        {"name": "pick 100 rays", "kind": "cast", "freq": 24, "rays": 100},
        # an object of a dynamic scene rebuilt each frame
        {"name": "build 6k", "kind": "build", "freq": 17, "builder": "lbvh", "meshes": 2, "index": "int32"},
        # the benchmark's scene loaded
        {"name": "build 1.3M", "kind": "build", "freq": 256, "builder": "lbvh", "meshes": 1, "index": "int32"},
        # a static scene built once with the better tree
        {"name": "build ploc 150k", "kind": "build", "freq": 87, "builder": "ploc", "meshes": 1, "index": "int32"},
        # the benchmark's step: a full HD frame's closest hits
        {"name": "camera 1080p 1.3M", "kind": "camera", "freq": 256, "width": 1920, "height": 1080},
        # incoherent closest hits through the largest scene
        {"name": "cast 1.5M random", "kind": "cast", "freq": 256, "rays": 1500000},
        # occlusion and visibility rays of bounded length through a middle scene
        {"name": "segments 2M", "kind": "segments", "freq": 112, "rays": 2000000},
        # a shaded full HD frame of the largest scene
        {"name": "render 1080p 1.3M", "kind": "render", "freq": 256, "width": 1920, "height": 1080,
         "texture": 512, "bilinear": True, "shadows": True},
        # a render server's queue: 48 views of 12 scenes
        {"name": "batch 48 views", "kind": "batch", "scenes": 12, "views": 4, "freq_lo": 7, "freq_hi": 150,
         "size_lo": 128, "size_hi": 768},
        # a quarter of a full HD path-traced frame
        {"name": "paths 960x540", "kind": "paths", "freq": 112, "width": 960, "height": 540, "spp": 4, "bounces": 2},
        # the benchmark's mesh imported without normals
        {"name": "normals 650k", "kind": "normals", "freq": 256, "index": "int32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "build", "camera", "cast", "cast", "segments", "render", "render", "batch",
                       "paths", "normals"])
    freq = _log_int(rng, 5, 256)  # 500 .. 1.31M triangles
    if kind == "build":
        ploc, meshes = rng.random() < 0.3, rng.randint(1, 4)
        most = (87 if ploc else 256) / math.sqrt(meshes)  # as many triangles in all as one mesh may have
        return {"kind": kind, "freq": _log_int(rng, 5, most), "builder": "ploc" if ploc else "lbvh",
                "meshes": meshes, "index": rng.choice(["int32", "none", "int64"])}
    if kind == "camera":
        return {"kind": kind, "freq": freq, "width": _log_int(rng, 64, 1920), "height": _log_int(rng, 64, 1080)}
    if kind == "cast":
        return {"kind": kind, "freq": freq, "rays": _log_int(rng, 1, 1500000)}
    if kind == "segments":
        return {"kind": kind, "freq": _log_int(rng, 5, 112), "rays": _log_int(rng, 1, 2000000)}
    if kind == "render":
        return {"kind": kind, "freq": freq, "width": _log_int(rng, 64, 1920), "height": _log_int(rng, 64, 1080),
                "texture": rng.choice([0, 33, 256, 512]), "bilinear": rng.random() < 0.7,
                "shadows": rng.random() < 0.8}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(1, 12), "views": rng.randint(1, 4), "freq_lo": 7,
                "freq_hi": _log_int(rng, 10, 150), "size_lo": _log_int(rng, 50, 128),
                "size_hi": _log_int(rng, 130, 768)}
    if kind == "paths":
        return {"kind": kind, "freq": _log_int(rng, 5, 112), "width": _log_int(rng, 64, 960),
                "height": _log_int(rng, 64, 540), "spp": rng.randint(1, 4), "bounces": rng.randint(0, 2)}
    return {"kind": kind, "freq": freq, "index": rng.choice(["int32", "none"])}


# ---- scenes ----

@functools.lru_cache(maxsize=64)
def _unit_sphere(freq):
    """Positions, triangles and texture coordinates of the undisplaced sphere."""
    pos, idx = scenes.geodesic_sphere(freq)
    return pos, idx, scenes.spherical_uv(pos)


def _displaced(freq, rng):
    """Vertex positions of a displaced sphere in the unit cube."""
    pos = _unit_sphere(freq)[0]
    r = 1.0 + 0.05 * rng.standard_normal(len(pos))
    return scenes.normalize_unit_cube(pos * r[:, None])


def _mesh(pos, idx, uv, index="int32"):
    """A Mesh on the device with computed normals; `index`: the type of its index buffer."""
    if index == "none":
        pos, uv, idx = pos[idx].reshape(-1, 3), uv[idx].reshape(-1, 2), None
    v = torch.from_numpy(np.ascontiguousarray(pos, np.float32)).cuda()
    t = torch.from_numpy(np.ascontiguousarray(uv, np.float32)).cuda()
    i = None if idx is None else torch.from_numpy(np.ascontiguousarray(idx, np.int32)).cuda()
    m = ren.mesh_from_tensors(v, i, uvs=t)
    if index == "int64":
        m.indices = ren.create_buffer_from(idx.astype(np.int64).reshape(-1))
    m.compute_normals()
    return m


def _sphere_meshes(freq, rng, count=1, index="int32", scale=1.0):
    """`count` displaced spheres side by side along x."""
    _, idx, uv = _unit_sphere(freq)
    out = []
    for k in range(count):
        pos = _displaced(freq, rng) * np.float32(scale)
        pos[:, 0] += 1.2 * (k - 0.5 * (count - 1))
        out.append(_mesh(pos, idx, uv, index))
    return out


def _ground():
    d = scenes.ground_plane()
    return _mesh(d["pos"], d["idx"], d["uv"])


def _scene(freq, rng):
    """The benchmark's kind of scene: one displaced sphere on a ground plane."""
    return _sphere_meshes(freq, rng) + [_ground()]


def _eye(rng, distance=3.0):
    """A view of the origin from a little above the horizon, from any side."""
    a, h = rng.uniform(0, 2 * math.pi), rng.uniform(0.0, 0.35)
    return (distance * math.cos(h) * math.sin(a), distance * math.sin(h), distance * math.cos(h) * math.cos(a))


def _camera(rng, width, height, distance=3.0):
    return ren.Camera(_eye(rng, distance), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), math.pi / 4, width / height)


def _random_rays(n, seed):
    """Origins in and around the sphere, directions uniform on the sphere."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    o = (torch.rand((n, 3), device="cuda", generator=g) * 2 - 1) * 0.6
    d = torch.randn((n, 3), device="cuda", generator=g)
    return o, d / d.norm(dim=1, keepdim=True)


# ---- one case ----

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "build":
        s["meshes"] = _sphere_meshes(case["freq"], rng, case["meshes"], case["index"])
        s["tuning"] = {"builder": case["builder"]}
    elif kind == "normals":
        _, idx, uv = _unit_sphere(case["freq"])
        s["mesh"] = _mesh(_displaced(case["freq"], rng), idx, uv, case["index"])
        s["out"] = torch.empty((s["mesh"].vertices.shape[0], 3), dtype=torch.float32, device="cuda")
    elif kind == "batch":
        lo, hi = math.log(case["freq_lo"]), math.log(case["freq_hi"])
        requests = []
        for k in range(case["scenes"]):
            freq = int(round(math.exp(lo + (hi - lo) * (k + 0.5) / case["scenes"])))
            rc = ren.Raycaster(_sphere_meshes(freq, rng))
            for v in range(case["views"]):
                f = (k * case["views"] + v + 0.5) / (case["scenes"] * case["views"])
                size = int(round(case["size_lo"] * (case["size_hi"] / case["size_lo"]) ** ((f * 7.0) % 1.0)))
                requests.append(RenderRequest(rc, _camera(rng, size, size), size, size))
        s["batch"] = BatchRender(requests)
    elif kind == "paths":
        # a row of three spheres on the ground, seen from above so that most paths bounce
        meshes = _sphere_meshes(case["freq"], rng, 3) + [_ground()]
        s["rc"] = ren.Raycaster(meshes)
        eye = (0.6 * rng.uniform(-1, 1), 1.2, 2.2)
        s["camera"] = ren.Camera(eye, (0.0, -0.3, 0.0), (0.0, 1.0, 0.0), math.pi / 4, case["width"] / case["height"])
        s["counts"] = torch.zeros(case["bounces"] + 1, dtype=torch.int32, device="cuda")
        s["seed"] = seed
    else:
        s["rc"] = ren.Raycaster(_scene(case["freq"], rng))
        if kind in ("camera", "render"):
            s["camera"] = _camera(rng, case["width"], case["height"])
        if kind == "render":
            size = case["texture"]
            s["textures"] = None
            if size:
                texels = rng.integers(0, 256, (size, size, 4), dtype=np.uint8)
                s["textures"] = TextureBinding([torch.from_numpy(texels).cuda()], [0, 0])
        if kind == "cast":
            o, d = _random_rays(case["rays"], seed)
            buf = ren.create_buffer(case["rays"], ren.Ray)
            f = buf.tensor(torch.float32, (case["rays"], 8))
            f.zero_()
            f[:, 0:3], f[:, 4:7] = o, d
            s["rays"] = buf
        if kind == "segments":
            a, _ = _random_rays(case["rays"], seed)
            b, _ = _random_rays(case["rays"], seed + 1000003)
            length = (b - a).norm(dim=1).clamp_min(1e-6)
            d = (b - a) / length[:, None]
            s["rays"] = {"ox": a[:, 0].contiguous(), "oy": a[:, 1].contiguous(), "oz": a[:, 2].contiguous(),
                         "dx": d[:, 0].contiguous(), "dy": d[:, 1].contiguous(), "dz": d[:, 2].contiguous(),
                         "tmax": length}
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "build":
        rc = ren.Raycaster(state["meshes"], tuning=state["tuning"])
        return {k: v.view(torch.int32) for k, v in rc.scene_arrays().items()}
    if kind == "normals":
        return ren.compute_normals(state["mesh"], out=state["out"])
    if kind == "batch":
        state["batch"].launch()
        return {"images": state["batch"].images, "stats": state["batch"].stats}
    if kind == "camera":
        return state["rc"].cast_camera(state["camera"], case["width"], case["height"])
    if kind == "cast":
        hits = state["rc"].ray_cast(state["rays"])
        n = case["rays"]
        return {"t_u_v": hits.tensor(torch.float32, (n, 5))[:, :3], "ids": hits.tensor(torch.int32, (n, 5))[:, 3:]}
    if kind == "segments":
        return state["rc"].occluded(state["rays"])
    if kind == "render":
        return state["rc"].render(state["camera"], case["width"], case["height"], textures=state["textures"],
                                  shadows=case["shadows"], bilinear=case["bilinear"])
    radiance = state["rc"].trace_paths(state["camera"], case["width"], case["height"], spp=case["spp"],
                                       bounces=case["bounces"], seed=state["seed"], counts=state["counts"])
    return {"radiance": radiance, "counts": state["counts"]}


def _sizes(case):
    """Triangles and vertices of the case's scene (of its spheres; the ground adds 2 and 4)."""
    f = case["freq"]
    return 20 * f * f, 10 * f * f + 2


def _ray_work(rays, tris, n_meshes=1):
    """One ray's least work is a box test of four children per level and one triangle test; a scene
    record is read at most once per scene, and only where there is a ray for it."""
    levels = max(1.0, math.log(max(tris, 2) / 4.0, 4.0))
    return min(tris, rays) * 48.0 + min(tris / 3.0, rays) * 128.0, rays * (levels * 4 * 18 + 50.0)


def work(case):
    kind = case["kind"]
    if kind == "build":
        t, v = _sizes(case)
        t, v = t * case["meshes"], v * case["meshes"]
        per_index = {"int32": 4, "int64": 8, "none": 0}[case["index"]]
        v = 3 * t if case["index"] == "none" else v
        # vertex records and indices in; nodes, 4-wide nodes, triangles, shading, keys, orders out
        return {"bytes": 80.0 * v + 3 * per_index * t + (64 + 128 + 48 + 64 + 12) * t, "flops": 60.0 * t}
    if kind == "normals":
        t, v = _sizes(case)
        if case["index"] == "none":
            return {"bytes": 24.0 * 3 * t, "flops": 60.0 * t}
        return {"bytes": 12.0 * t + 24.0 * v, "flops": 40.0 * t + 20.0 * v}
    if kind == "batch":
        b = f = 0.0
        lo, hi = math.log(case["freq_lo"]), math.log(case["freq_hi"])
        for k in range(case["scenes"]):
            freq = int(round(math.exp(lo + (hi - lo) * (k + 0.5) / case["scenes"])))
            for v in range(case["views"]):
                at = (k * case["views"] + v + 0.5) / (case["scenes"] * case["views"])
                size = int(round(case["size_lo"] * (case["size_hi"] / case["size_lo"]) ** ((at * 7.0) % 1.0)))
                wb, wf = _ray_work(size * size * 0.3, 20 * freq * freq)  # a sphere fills a third of its image
                b, f = b + wb + 12.0 * size * size, f + wf * 1.5
        return {"bytes": b, "flops": f}
    t = _sizes(case)[0]
    if kind == "paths":
        n = case["width"] * case["height"] * case["spp"]
        b, f = _ray_work(n * (1 + 0.6 * case["bounces"]), 3 * t)
        return {"bytes": b + 4.0 * case["width"] * case["height"], "flops": f}
    if kind == "cast":
        b, f = _ray_work(case["rays"], t)
        return {"bytes": b + (32 + 20) * case["rays"], "flops": f}
    if kind == "segments":
        b, f = _ray_work(case["rays"], t)
        return {"bytes": b + (28 + 1) * case["rays"], "flops": f}
    n = case["width"] * case["height"]
    if kind == "camera":
        b, f = _ray_work(n, t)
        return {"bytes": b + 16.0 * n, "flops": f}
    b, f = _ray_work(n * (1.4 if case["shadows"] else 1.0), t)
    return {"bytes": b + 12.0 * n + 4.0 * case["texture"] ** 2 + 64.0 * min(n, t), "flops": f}


# ---- 64-bit values of the smaller cases, from the definitions alone ----

_MOST_PAIRS = 3e10


def _triangles64(freq, rng):
    """v0, v1, v2 of every triangle of _scene(freq, rng), the sphere's first."""
    pos, idx = _displaced(freq, rng), _unit_sphere(freq)[1]
    g = scenes.ground_plane()
    tri = np.concatenate([pos[idx], g["pos"][g["idx"]]]).astype(np.float64)
    return torch.from_numpy(tri).cuda()


def _closest64(o, d, tri, tmin=0.0, skip=None):
    """t, u, v and triangle of each ray's closest hit by Moller and Trumbore's equations over every pair."""
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    n = torch.linalg.cross(e1, e2)
    an = (a * n).sum(1)
    ae1, ae2 = torch.linalg.cross(a, e1), torch.linalg.cross(a, e2)
    step = max(1, int(6e7 // len(tri)))
    out = []
    for k in range(0, len(o), step):
        oo, dd = o[k:k + step], d[k:k + step]
        od = torch.linalg.cross(oo, dd)
        det = -(dd @ n.T)
        # (o - a) . (d x e2) = (o x d) . e2 + d . (a x e2); the same for e1 with the other sign
        u = (od @ e2.T + dd @ ae2.T) / det
        v = -(od @ e1.T + dd @ ae1.T) / det
        t = (oo @ n.T - an) / det
        ok = (det != 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > tmin)
        if skip is not None:
            ok &= torch.arange(len(tri), device=o.device)[None, :] != skip[k:k + step, None]
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, at = t.min(1)
        hit = torch.isfinite(best)
        w = torch.zeros_like(best)
        out.append((best, torch.where(hit, u.gather(1, at[:, None])[:, 0], w),
                    torch.where(hit, v.gather(1, at[:, None])[:, 0], w),
                    torch.where(hit, at, torch.full_like(at, -1))))
    return [torch.cat(x) for x in zip(*out)]


def _camera_rays64(eye, width, height):
    """Pixel-centre rays of a 45 degree look_at camera on the origin."""
    eye = np.asarray(eye, np.float64)
    z = -eye / np.linalg.norm(eye)
    x = np.cross([0.0, 1.0, 0.0], z)
    x /= np.linalg.norm(x)
    y = np.cross(z, x)
    th = math.tan(math.pi / 8)
    nx = (np.arange(width) + 0.5) / width * 2 - 1
    ny = 1 - (np.arange(height) + 0.5) / height * 2
    d = (nx[None, :, None] * x * th * width / height + ny[:, None, None] * y * th + z).reshape(-1, 3)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return torch.from_numpy(np.broadcast_to(eye, d.shape).copy()).cuda(), torch.from_numpy(d).cuda()


def _normals64(pos, idx):
    p = torch.from_numpy(pos).cuda().double()
    i = torch.from_numpy(idx).cuda().long()
    fn = torch.linalg.cross(p[i[:, 1]] - p[i[:, 0]], p[i[:, 2]] - p[i[:, 0]])
    n = torch.zeros_like(p)
    for k in range(3):
        n.index_add_(0, i[:, k], fn)
    return n / n.norm(dim=1, keepdim=True).clamp_min(1e-300)


def _texture64(texels, uv, bilinear):
    """OpenCL's linear filter with repeat addressing, or the nearest texel, of RGBA8 texels."""
    h, w = texels.shape[:2]
    s = uv - torch.floor(uv)
    tex = texels[..., :3].double() / 255.0
    if not bilinear:
        i = (s[:, 0] * w).long().clamp_max(w - 1)
        j = (s[:, 1] * h).long().clamp_max(h - 1)
        return tex[j, i]
    x, y = s[:, 0] * w - 0.5, s[:, 1] * h - 0.5
    i0, j0 = torch.floor(x), torch.floor(y)
    a, b = (x - i0)[:, None], (y - j0)[:, None]
    i0, j0 = i0.long() % w, j0.long() % h
    i1, j1 = (i0 + 1) % w, (j0 + 1) % h
    return (tex[j0, i0] * (1 - a) + tex[j0, i1] * a) * (1 - b) + (tex[j1, i0] * (1 - a) + tex[j1, i1] * a) * b


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "normals":
        pos, idx = _displaced(case["freq"], rng), _unit_sphere(case["freq"])[1]
        if case["index"] == "none":
            pos, idx = pos[idx].reshape(-1, 3), np.arange(3 * len(idx)).reshape(-1, 3)
        return _normals64(np.ascontiguousarray(pos, np.float32), idx)
    if kind not in ("camera", "cast", "render"):
        return None
    rays = case["rays"] if kind == "cast" else case["width"] * case["height"]
    if rays * (_sizes(case)[0] + 2) > _MOST_PAIRS:
        return None
    tri = _triangles64(case["freq"], rng)
    if kind == "cast":
        o, d = _random_rays(rays, seed)
        t, u, v, _ = _closest64(o.double(), d.double(), tri)
        return {"t_u_v": torch.stack([t, u, v], 1), "ids": None}
    width, height = case["width"], case["height"]
    o, d = _camera_rays64(_eye(rng), width, height)
    t, u, v, at = _closest64(o, d, tri)
    if kind == "camera":
        return {"t": t, "u": u, "v": v, "prim": None}
    # Lambert with the interpolated normal, 0.2 ambient, one shadow ray, one texture for both meshes
    pos, (_, idx, uv) = _displaced(case["freq"], np.random.default_rng(seed)), _unit_sphere(case["freq"])
    g = scenes.ground_plane()
    nrm = _normals64(pos, idx)
    idx_d = torch.from_numpy(idx).cuda().long()
    corner_n = torch.cat([nrm[idx_d], torch.from_numpy(g["nrm"][g["idx"]]).cuda().double()])
    corner_uv = torch.from_numpy(np.concatenate([uv[idx], g["uv"][g["idx"]]])).cuda().double()
    hit = at >= 0
    k, w = at.clamp_min(0), torch.stack([1 - u - v, u, v], 1)[:, :, None]
    n = (corner_n[k] * w).sum(1)
    light = torch.from_numpy(LIGHT).cuda()
    ndl = ((n / n.norm(dim=1, keepdim=True)) @ light).clamp_min(0.0)
    lit = hit & (ndl > 0)
    free = torch.ones_like(ndl)
    if case["shadows"]:
        so = o[lit] + t[lit][:, None] * d[lit]
        blocked = _closest64(so, light.expand_as(so), tri, tmin=1e-4, skip=at[lit])[3] >= 0
        free[lit] = torch.where(blocked, 0.0, 1.0).double()
    shade = (0.2 + free * ndl)[:, None].expand(-1, 3)
    if case["texture"]:
        texels = rng.integers(0, 256, (case["texture"], case["texture"], 4), dtype=np.uint8)
        shade = shade * _texture64(torch.from_numpy(texels).cuda(), (corner_uv[k] * w).sum(1), case["bilinear"])
    return torch.where(hit[:, None], shade, torch.zeros_like(shade)).reshape(height, width, 3)
