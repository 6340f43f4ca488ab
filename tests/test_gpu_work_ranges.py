"""Rays that a persistent trace hands out from its work counters: launches with
far more rays than one range per wave, an odd remainder, refills of every size
into lanes whose result is not stored yet, the split stack, and launches one
after the other on the same counters.  Every ray's result equals the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,waves", [
    (100_003, 1),  # first ranges and chunks of one ray per lane
    (100_003, 2),
    (400_037, 1),  # first ranges of half a share, chunks of two rays per lane
])
def test_every_ray_once(gpu_ctx, oracle, n, waves):
    import torch

    share = n // (torch.cuda.get_device_properties(0).multi_processor_count * waves)
    assert share > 64 and (share >= 512) == (n > 400_000)
    s = scenes.spheres(n_spheres=4)
    gpu_ctx.upload_scene(s)
    gpu_ctx.rebuild_nmh()
    tree = s.vertices[gpu_ctx.read_permutation()]
    rays = scenes.incoherent_rays(n, 0.0, 100.0, seed=23)
    shadow = rays.copy()
    shadow[:, 3] = np.random.default_rng(24).uniform(1.0, 60.0, n).astype(np.float32)
    ids_o, tuv_o = oracle.trace(tree, rays)
    any_o, _ = oracle.trace(tree, shadow, any_hit=True)
    want = np.concatenate([ids_o[:, None], tuv_o.view(np.int32)], axis=1)
    assert (ids_o >= 0).any() and (any_o >= 0).any()
    rays, shadow = torch.from_numpy(rays).cuda(), torch.from_numpy(shadow).cuda()
    try:
        for block in (64, 128, 256):
            for refill in (1, 7, 64):
                for rows in (0, 3):
                    gpu_ctx.set_trace_params(block=block, refill=refill, waves_per_cu=waves, stack_lds_rows=rows)
                    hits = torch.full((2, n, 4), -7, dtype=torch.int32, device="cuda")
                    ids = torch.full((2, n), -7, dtype=torch.int32, device="cuda")
                    torch.cuda.synchronize()
                    for k in range(2):
                        gpu_ctx.trace_closest_ptr(n, rays.data_ptr(), hits[k].data_ptr())
                        gpu_ctx.trace_any_ptr(n, shadow.data_ptr(), ids[k].data_ptr())
                    gpu_ctx.synchronize()
                    for k in range(2):
                        assert np.array_equal(hits[k].cpu().numpy(), want), (block, refill, rows, k)
                        assert np.array_equal(ids[k].cpu().numpy(), any_o), (block, refill, rows, k)
    finally:
        gpu_ctx.set_trace_params()
