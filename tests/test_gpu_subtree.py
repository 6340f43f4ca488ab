"""The LDS subtree phase of the build (groups of at most 4096 triangles): the
tree equals the oracle's at the sizes where its levels, sort slots and node
counts change, with distinct keys and with keys of which most are equal (the
sort must be stable and the first maximum the lowest position)."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [None, 0.5, 20.0])
@pytest.mark.parametrize("count", [2, 4, 6, 8, 126, 128, 130, 1022, 1024, 2044, 2046, 2048, 2050, 2052, 4094, 4096, 4098,
                                   5000, 8190, 16_384, 70_002])
def test_subtree_equals_oracle(gpu_ctx, oracle, count, grid):
    s = scenes.random_soup(seed=count, n=count, grid=grid)
    gpu_ctx.upload_geometry(s.vertices, s.normals, s.texcoords, s.shader_ids)
    gpu_ctx.rebuild_nmh()
    assert np.array_equal(gpu_ctx.read_permutation(), oracle.nmh_build(s.vertices))
