"""Trees of one to four levels: up to three they are traced by one lane per ray with
both triangles of each node tested exactly, above that by waves with the reject
test.  Hits equal the oracle's for every launch shape, ray counts at the edges of a
wave and a block, and rays that no shortcut serves."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [2, 4, 6, 12, 14, 16, 30])
def test_hits(gpu_ctx, oracle, count):
    v = scenes.random_soup(seed=count, n=count, box=4.0).vertices
    gpu_ctx.upload_geometry(v)
    gpu_ctx.rebuild_nmh()
    tree = v[gpu_ctx.read_permutation()]
    rays = scenes.incoherent_rays(20_003, -1.0, 5.0, seed=count)
    # half of them toward a triangle's centroid, from its front as often as not
    c = v.reshape(-1, 3, 3).mean(axis=2)[np.random.default_rng(count).integers(0, count, 10_000)]
    d = c - rays[:10_000, 0:3]
    rays[:10_000, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:300:3, 4:7] = (0.0, -0.0, 1.0)
    rays[1:300:3, 4] = 0.0
    rays[300:400, 4:7] *= np.float32(1000.0)
    rays[400:403, 0], rays[403:406, 5], rays[406:409, 6] = np.nan, np.inf, np.nan
    rays[500:600, 3] = np.float32(0.5)
    ids_o, tuv_o = oracle.trace(tree, rays)
    any_o, _ = oracle.trace(tree, rays, any_hit=True)
    assert (ids_o >= 0).sum() > 100
    try:
        for p in (dict(), dict(persistent=0, block=64), dict(persistent=0, block=256), dict(waves_per_cu=1),
                  dict(block=64, stack_lds_rows=1)):
            gpu_ctx.set_trace_params(**p)
            for n in (1, 63, 65, 257, rays.shape[0]):
                ids_g, tuv_g = gpu_ctx.trace(rays[:n])
                assert np.array_equal(ids_g, ids_o[:n]), (p, n)
                assert np.array_equal(tuv_g.view(np.uint32), tuv_o[:n].view(np.uint32)), (p, n)
                any_g, _ = gpu_ctx.trace(rays[:n], any_hit=True)
                assert np.array_equal(any_g, any_o[:n]), (p, n)
    finally:
        gpu_ctx.set_trace_params()
