"""Builds on both sides of the size from which records are stored past the caches, byte for byte against the
twin."""
import numpy as np
import pytest

from helpers import gpu_from_meshes, twin_from_meshes
from test_gpu_parity import assert_build_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [499999, 500000])
def test_store_line(ren, n):
    rng = np.random.default_rng(n)
    pos = (rng.uniform(-1, 1, (n, 1, 3)) + 1e-3 * rng.uniform(-1, 1, (n, 3, 3))).reshape(-1, 3).astype(np.float32)
    meshes = [{"pos": pos, "idx": np.arange(3 * n, dtype=np.int32).reshape(-1, 3)}]
    assert_build_equal(gpu_from_meshes(meshes), twin_from_meshes(meshes))
