"""Groups of lanes on what they are not timed on: stacks past the switch to single entries, and rays with NaN,
infinite, zero and denormal components, against the oracle and the one-lane walks."""
import numpy as np
import pytest
import torch

from helpers import deep_wide_scene, gpu_from_meshes, soa_tensors, twin_from_meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [400, 9000])  # 64 and 16 lanes per ray
def test_stacks_past_the_switch(ren, n):
    """test_oracle_group_stack shows that these stacks pass the switch."""
    meshes = deep_wide_scene()
    rc, tw = gpu_from_meshes(meshes), twin_from_meshes(meshes)
    rng = np.random.default_rng(n)
    o, d = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    o[::3] = (3.5, -2.5, 0.5)  # beyond the last plane: these enter every box and hit nothing
    d[::3] = (1.0, -1.0, 0.0) + rng.uniform(-0.2, 0.2, (len(d[::3]), 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o, d = o.astype(np.float32), d.astype(np.float32)
    rays = soa_tensors(o, d)
    _, prim = tw.brute_closest32(o, d)
    assert (prim[::3] == -1).all() and (prim >= 0).sum() > n // 4
    np.testing.assert_array_equal(rc.trace_soa(rays)["prim"].cpu().numpy(), prim)
    np.testing.assert_array_equal(rc.occluded(rays).cpu().numpy(), prim >= 0)


@pytest.fixture(scope="module")
def plain(ren):
    from rendertoy_amd import scenes
    meshes = [scenes.icosphere(20, 5), scenes.ground_plane()]
    return gpu_from_meshes(meshes), twin_from_meshes(meshes)


def test_special_rays(plain):
    """Every walk gives such a ray the oracle's hit, and a miss where it has NaN anywhere."""
    rc, tw = plain
    rng = np.random.default_rng(5)
    special = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e-40, -1e-40, 3e38, -3e38], np.float32)
    n = 6000
    o = rng.uniform(-1.5, 1.5, (n, 3)).astype(np.float32)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    for a in (o, d):
        put = rng.random((n, 3)) < 0.25
        a[put] = rng.choice(special, put.sum())
    ref = tw.trace_closest(o, d)
    occluded = tw.trace_any(o, d)
    nan = np.isnan(o).any(1) | np.isnan(d).any(1)
    assert (ref["prim"][nan] == -1).all() and (ref["prim"] >= 0).sum() > 200
    for count in (300, n, 70000):  # 64 and 16 lanes per ray, one
        k = np.arange(count) % n
        rays = soa_tensors(o[k], d[k])
        for tuning in (None, {"query": "binary"}):
            hits = rc.trace_soa(rays, tuning=tuning)
            for f in ("prim", "t", "u", "v"):
                np.testing.assert_array_equal(hits[f].cpu().numpy().view(np.uint32), ref[f][k].view(np.uint32))
            np.testing.assert_array_equal(rc.occluded(rays, tuning=tuning).cpu().numpy(), occluded[k])


def test_special_intervals(plain):
    rc, tw = plain
    rng = np.random.default_rng(6)
    n = 70000
    o = rng.uniform(-1.5, 1.5, (n, 3)).astype(np.float32)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    values = np.array([np.nan, np.inf, -np.inf, 0.0, -1.0, -0.5, 0.5, 1.0, 3e38, -3e38], np.float32)
    rays = soa_tensors(o, d)
    lo, hi = rng.choice(values, n), rng.choice(values, n)
    rays["tmin"], rays["tmax"] = torch.from_numpy(lo).cuda(), torch.from_numpy(hi).cuda()
    one = rc.trace_soa(rays)
    blocked = rc.occluded(rays)
    assert int((one["prim"] >= 0).sum()) > 1000
    for a, b in ((0, 300), (300, 6300), (6300, 66300)):
        part = {k: v[a:b].contiguous() for k, v in rays.items()}
        for tuning in (None, {"query": "binary"}, {"lane_stack": 31}):
            hits = rc.trace_soa(part, tuning=tuning)
            assert torch.equal(hits["prim"], one["prim"][a:b])
            assert torch.equal(rc.occluded(part, tuning=tuning), blocked[a:b])
    empty = np.isnan(lo) | np.isnan(hi) | ~(lo < hi)
    assert (one["prim"].cpu().numpy()[empty] == -1).all() and not blocked.cpu().numpy()[empty].any()

