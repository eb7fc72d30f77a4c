"""Hits of ray buffers do not depend on how many rays the call has, on either side of the sizes at which the
one-lane walks fetch whole leaves or only their triangles."""
import pytest
import torch

from helpers import gpu_from_meshes, random_rays, soa_tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("freq,n", [(60, 262144), (82, 524288), (20, 524289)])
def test_split_buffers(ren, freq, n):
    from rendertoy_amd import scenes
    rc = gpu_from_meshes([scenes.icosphere(freq, 4), scenes.ground_plane()])
    rays = soa_tensors(*random_rays(n, freq))
    occ, hits = rc.occluded(rays), rc.trace_soa(rays)
    cut = n - 140000
    for a, b in ((0, cut), (cut, n)):
        part = {k: v[a:b].contiguous() for k, v in rays.items()}
        assert torch.equal(rc.occluded(part), occ[a:b])
        for k, v in rc.trace_soa(part).items():
            assert torch.equal(v.view(torch.int32), hits[k][a:b].view(torch.int32)), k
