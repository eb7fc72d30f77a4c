"""Batches handed out from the tile queues take no longer than from the single counter, whatever the images'
widths and the number of jobs, and render the same images."""
import numpy as np
import pytest
import torch

from helpers import gpu_from_meshes

pytestmark = pytest.mark.gpu


def _sphere():
    from rendertoy_amd import scenes
    return [scenes.icosphere(8, 3), scenes.ground_plane()]


def _random_triangles():
    rng = np.random.default_rng(50000)
    s = 50000 ** (-1 / 3)
    pos = (rng.uniform(-0.7, 0.7, (50000, 1, 3)) + rng.uniform(-s, s, (50000, 3, 3))).reshape(-1, 3).astype(np.float32)
    return [{"pos": pos, "idx": np.arange(150000, dtype=np.int32).reshape(-1, 3), "nrm": None, "uv": None}]


def _time(f):
    f()
    times = []
    for _ in range(9):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(200000)  # the launches queue up behind it
        a.record()
        f()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


@pytest.mark.parametrize("scene,jobs,lo,hi", [(_sphere, 8, 1024, 1024), (_sphere, 64, 256, 256), (_sphere, 1, 500, 500),
                                              (_random_triangles, 64, 256, 256), (_random_triangles, 300, 32, 128),
                                              (_random_triangles, 2000, 16, 40)])
def test_queues_take_no_longer(ren, scene, jobs, lo, hi):
    from rendertoy_amd import _native as N
    from rendertoy_amd.batch import BatchRender, RenderRequest
    rc, rng = gpu_from_meshes(scene()), np.random.default_rng(jobs)
    reqs = []
    for _ in range(jobs):
        size = int(rng.integers(lo, hi + 1))
        eye = np.array((0.6, 0.8, 2.2)) * rng.uniform(0.8, 1.2, 3)
        reqs.append(RenderRequest(rc, ren.Camera(tuple(eye), (0, 0, 0), (0, 1, 0), 0.785, 1.0), size, size))
    batch = BatchRender(reqs)
    queues = _time(batch.launch)
    images = [im.clone() for im in batch.images]
    batch.workspace = batch.workspace[:4 * (64 + jobs + 1)]  # no room for the queues
    counter = _time(batch.launch)
    assert all(torch.equal(a, b) for a, b in zip(images, batch.images))
    assert queues < 1.15 * counter, (queues, counter)


@pytest.mark.parametrize("jobs", [1, 5, 63])
def test_reported_size_reaches_the_queues(ren, jobs):
    """A workspace of rt_render_batch_queue_bytes is handed out from the queues, one byte less is not."""
    import ctypes
    from rendertoy_amd import _native as N
    from rendertoy_amd.batch import BatchRender, RenderRequest
    lib, rc = N.load(), gpu_from_meshes(_sphere())
    cam = ren.Camera((0.6, 0.8, 2.2), (0, 0, 0), (0, 1, 0), 0.785, 1.0)
    batch = BatchRender([RenderRequest(rc, cam, 40, 40)] * jobs)
    size, cfg = lib.rt_render_batch_queue_bytes(jobs), batch.config.to_c()
    assert batch.workspace.numel() >= size > lib.rt_render_batch_workspace_bytes(jobs)
    for given in (size, size - 1):
        ws = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device="cuda")
        N.check(lib.rt_render_batch(batch.jobs_dev.data_ptr(), jobs, ctypes.byref(cfg), ws.data_ptr(), given,
                                    N.stream_handle()), "rt_render_batch")
        past = ws[lib.rt_render_batch_workspace_bytes(jobs):size]
        assert bool((past != 0x5A).any()) == (given == size)
        assert bool((ws[size:] == 0x5A).all())
