"""Batches whose workspace has room for the tile queues: the images, hits and counts are those of the
single counter, at every number of queues in use and with jobs that have no tiles."""
import ctypes
import math

import numpy as np
import pytest
import torch

from helpers import camera, gpu_from_meshes

pytestmark = pytest.mark.gpu


def _run(N, lib, jobs, n, cfg, extra):
    ws = torch.full((lib.rt_render_batch_workspace_bytes(n) + extra,), 0xA5, dtype=torch.uint8, device="cuda")
    N.check(lib.rt_render_batch(jobs.data_ptr(), n, ctypes.byref(cfg), ws.data_ptr(), ws.numel(), N.stream_handle()),
            "rt_render_batch")
    torch.cuda.synchronize()
    return int(ws[4:8].view(torch.int32).item())


@pytest.mark.parametrize("sizes,grab,waves", [(((1, 1),), 4, 16), (((8, 8), (9, 8)), 64, 1),
                                              (((64, 64), (3, 200), (65, 7)), 1, 32),
                                              (tuple((8 + 5 * k, 97 - k) for k in range(70)), 4, 16)])
def test_queues_equal_the_single_counter(ren, sizes, grab, waves):
    from rendertoy_amd import _native as N, scenes
    from rendertoy_amd.batch import BatchConfig, BatchRender, RenderRequest
    lib = N.load()
    pool = [gpu_from_meshes([scenes.icosphere(f, 50 + f), scenes.ground_plane()]) for f in (3, 20, 3, 9)]
    pool.append(ren.Raycaster([]))
    reqs = [RenderRequest(pool[k % len(pool)], camera(eye=(0.3 * math.sin(k), 0.4, 2.0), aspect=w / h), w, h,
                          return_hits=True) for k, (w, h) in enumerate(sizes)]
    b = BatchRender(reqs, config=BatchConfig(waves_per_cu=waves, tiles_per_grab=grab))
    n, cfg = b.n_jobs, b.config.to_c()
    jobs = (N.rt_render_job * n).from_buffer_copy(b.jobs_dev.cpu().numpy().tobytes())
    if n > 2:
        jobs[1].out.rgb = None  # skipped with status 2
    dev = torch.frombuffer(bytearray(bytes(jobs)), dtype=torch.uint8).cuda()
    results = []
    for extra in (0, 16640 + 4 * n - 4 - 256, 16640 + 4 * n, 1 << 20):
        for im, h in zip(b.images, b.hits):
            im.fill_(-1.0), h["t"].fill_(-1.0), h["prim"].fill_(-9)
        b.stats.fill_(-1)
        assert _run(N, lib, dev, n, cfg, extra) == (2 if n > 2 else 0)
        results.append([x.clone() for im, h in zip(b.images, b.hits)
                        for x in (im.view(torch.int32), h["t"].view(torch.int32), h["prim"])] + [b.stats.clone()])
    for other in results[1:]:
        assert all(torch.equal(x, y) for x, y in zip(results[0], other))
    for k, r in enumerate(reqs):
        if n > 2 and k == 1:
            assert bool((b.images[k] == -1.0).all())
            continue
        alone = r.raycaster.render(r.camera, r.width, r.height)
        np.testing.assert_array_equal(b.images[k].cpu().numpy(), alone.cpu().numpy())
