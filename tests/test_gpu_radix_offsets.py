"""The build's radix levels: the output offsets that every tile sums from the
counts of its group's chunks (32 tiles of 2048 triangles) and of the tiles
before it, with few tiles, at the edges of a chunk, with several chunks, and
with groups of more than 64 chunks, whose sums have a launch of their own.  The
grid rounds the coordinates, so that most keys are equal and a group needs
fewer passes.  The tree equals the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,grid", [(4100, None), (6146, 20.0), (65_534, None), (65_538, 20.0), (131_072, None),
                                        (131_076, 0.5), (400_002, None), (4_300_002, None), (4_300_002, 20.0)])
def test_radix_levels_equal_oracle(gpu_ctx, oracle, count, grid):
    s = scenes.random_soup(seed=count, n=count, grid=grid)
    gpu_ctx.upload_geometry(s.vertices, s.normals, s.texcoords, s.shader_ids)
    gpu_ctx.rebuild_nmh()
    assert np.array_equal(gpu_ctx.read_permutation(), oracle.nmh_build(s.vertices))
