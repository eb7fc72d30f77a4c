"""Vertex normals at every length of run the kernels put in order differently (8 by a network, 64 by
selection, 4,096 in LDS, longer from the index list), and over the scan's chunks, against the twin."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(ren, pos, idx):
    import oracle
    m = ren.mesh_from_arrays(pos, idx)
    out = torch.empty((len(pos), 3), dtype=torch.float32, device="cuda")
    ren.compute_normals(m, out=out)
    want = np.ascontiguousarray(oracle.vertex_normals(pos, idx), np.float32)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("tris", [1, 8, 9, 63, 64, 65, 4096, 4097, 9000])
def test_fan(ren, tris):
    """Vertex 0 in every triangle, at a corner that changes; one more vertex in all of them by clamping."""
    rng = np.random.default_rng(tris)
    pos = rng.uniform(-1, 1, (tris + 3, 3)).astype(np.float32)
    idx = rng.integers(1, tris + 2, (tris, 3)).astype(np.int32)
    idx[np.arange(tris), rng.integers(0, 3, tris)] = 0
    _check(ren, pos, idx)
    idx[:, 1] = 10 ** 9
    _check(ren, pos, idx)


@pytest.mark.parametrize("verts", [2047, 2048, 2049, 2048 * 1024, 2048 * 1024 + 1])
def test_chunks(ren, verts):
    rng = np.random.default_rng(verts)
    pos = rng.uniform(-1, 1, (verts, 3)).astype(np.float32)
    idx = rng.integers(0, verts, (20000, 3)).astype(np.int32)
    idx[0] = [0, verts // 2, verts - 1]
    _check(ren, pos, idx)
