"""LBVH builds around the tree's block of 1,024 slots, byte for byte against the twin: spread triangles,
equal codes (every split by slot number), and codes in a few crowded cells."""
import numpy as np
import pytest

from helpers import gpu_arrays, gpu_from_meshes, twin_from_meshes
from test_gpu_parity import assert_build_equal

pytestmark = pytest.mark.gpu


def _mesh(n, kind):
    rng = np.random.default_rng(n)
    at = rng.uniform(-1, 1, (n, 1, 3))
    if kind == "equal":
        at[:] = 0.25
    elif kind == "crowded":
        at = np.sign(at) * 2.0 ** -np.floor(rng.exponential(4.0, (n, 1, 1)))
    size = 0.0 if kind == "equal" else 1e-3
    pos = at + size * rng.uniform(-1, 1, (n, 3, 3)) + (0.0 if size else np.eye(3))
    return {"pos": pos.reshape(-1, 3).astype(np.float32), "idx": np.arange(3 * n, dtype=np.int32).reshape(-1, 3)}


@pytest.mark.parametrize("kind", ["spread", "equal", "crowded"])
@pytest.mark.parametrize("n", [2, 5, 1023, 1024, 1025, 2047, 2048, 2049, 65 * 1024 + 1, 70 * 1024])
def test_block_edges(ren, n, kind):
    meshes = [_mesh(n, kind)]
    assert_build_equal(gpu_from_meshes(meshes), twin_from_meshes(meshes))


@pytest.mark.parametrize("kind", ["spread", "equal", "crowded"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 16384, 16385, 32767, 32768, 32769, 40961])
def test_small_order(ren, n, kind):
    """Order by chunks of 256 and merge by search (up to 32,768 triangles), and by radix passes from there."""
    meshes = [_mesh(n, kind)]
    assert_build_equal(gpu_from_meshes(meshes), twin_from_meshes(meshes))


def _ploc(ren, mesh):
    got = ren.Raycaster([ren.mesh_from_arrays(mesh["pos"], mesh["idx"])], tuning={"builder": "ploc"})
    return got, twin_from_meshes([mesh], builder="ploc")


@pytest.mark.parametrize("kind", ["spread", "equal", "crowded"])
@pytest.mark.parametrize("n", [2, 3, 64, 65, 129, 257, 513, 1025, 2048, 2049, 2305, 4097, 9000])
def test_ploc_sizes(ren, n, kind):
    """PLOC at the widths of a search in its last workgroup, at the hand-over to it (2,048 clusters) and at
    the tiles before it."""
    assert_build_equal(*_ploc(ren, _mesh(n, kind)))


@pytest.mark.parametrize("n", [40, 700])
def test_ploc_nan(ren, n):
    """Most boxes NaN: a search keeps its first candidate. A NaN's bits are not compared."""
    mesh = _mesh(n, "spread")
    mesh["pos"][np.random.default_rng(n).random(len(mesh["pos"])) < 0.9] = np.nan
    rc, tw = _ploc(ren, mesh)
    g = gpu_arrays(rc)
    np.testing.assert_array_equal(g["order"].view(np.uint32), tw.order)
    nodes, want = g["nodes"], np.asarray(tw.nodes).reshape(g["nodes"].shape)
    np.testing.assert_array_equal(np.ascontiguousarray(nodes[:, 12:14]).view(np.uint32),
                                  np.ascontiguousarray(want[:, 12:14]).view(np.uint32))
    np.testing.assert_array_equal(nodes[:, :12], want[:, :12])
