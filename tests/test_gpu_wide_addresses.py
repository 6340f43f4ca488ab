"""Trees of 2^26 nodes and more take 64-bit record addresses.  A small tree that is
made to take them gives the hits of the oracle and the frames that it gives with
32-bit offsets, bit for bit, with every stack row in LDS and with the split stack."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import native, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture()
def wide_ctx(gpu_ctx):  # gpu_ctx: torch's HIP runtime is loaded first
    with native.Context(0) as ctx:
        s = scenes.spheres(n_spheres=6, width=70, height=50)
        ctx.upload_scene(s)
        ctx.rebuild_nmh()
        yield ctx, s


@pytest.mark.parametrize("rows", [0, 3])
def test_traces(wide_ctx, oracle, rows):
    ctx, s = wide_ctx
    n = 100_003
    ctx.set_wide_records(True)
    ctx.set_trace_params(waves_per_cu=1, stack_lds_rows=rows)
    tree = s.vertices[ctx.read_permutation()]
    rays = scenes.incoherent_rays(n, 0.0, 100.0, seed=5)
    ids_g, tuv_g = ctx.trace(rays)
    ids_o, tuv_o = oracle.trace(tree, rays)
    assert (ids_o >= 0).any()
    assert np.array_equal(ids_g, ids_o)
    assert np.array_equal(tuv_g.view(np.uint32), tuv_o.view(np.uint32))
    rays[:, 3] = np.random.default_rng(6).uniform(1.0, 60.0, n).astype(np.float32)
    any_g, _ = ctx.trace(rays, any_hit=True)
    any_o, _ = oracle.trace(tree, rays, any_hit=True)
    assert np.array_equal(any_g, any_o)


@pytest.mark.parametrize("rows", [0, 3])
@pytest.mark.parametrize("mode,graph", [(native.MODE_PBR, 0), (native.MODE_PBR, 1), (native.MODE_COMPAT, 0)])
def test_frames(wide_ctx, mode, graph, rows):
    ctx, s = wide_ctx
    images = []
    for wide in (False, True):
        ctx.set_wide_records(wide)
        ctx.set_render_params(70 * 50 * 2, graph, 0, rows)
        ctx.frame_create(70, 50, 6)
        ctx.frame_render(s.camera, native.Context.opts(mode, 6, 4, 3, 5))
        images.append(ctx.frame_read())
    assert images[0][:, :3].max() > 0
    assert np.array_equal(images[0].view(np.uint32), images[1].view(np.uint32))


def test_switch_is_checked(wide_ctx):
    ctx, _ = wide_ctx
    assert ctx._lib.aur_set_wide_records(ctx.handle, 2) != native.AUR_OK
    assert ctx._lib.aur_set_wide_records(None, 0) != native.AUR_OK
