"""Traces recorded into a HIP graph share no state with the context's other
launches: replays on another stream, beside traces queued on the context's own,
give the hits that each launch gives alone.  One wave per CU, so that every
launch hands out most of its rays from its work counters."""
from __future__ import annotations

import numpy as np
import pytest

from aurora_amd import native, scenes

pytestmark = pytest.mark.gpu

N = 200_003


@pytest.fixture()
def setup(gpu_ctx, oracle):
    import torch

    s = scenes.spheres(n_spheres=10)
    with native.Context(0) as ctx:
        ctx.upload_scene(s)
        ctx.rebuild_nmh()
        ctx.set_trace_params(waves_per_cu=1)
        assert N > torch.cuda.get_device_properties(0).multi_processor_count * 64 * 4
        tree = s.vertices[ctx.read_permutation()]
        rays = [scenes.incoherent_rays(N, 0.0, 100.0, seed=k) for k in (1, 2)]
        want = [np.concatenate([ids[:, None], tuv.view(np.int32)], axis=1)
                for ids, tuv in (oracle.trace(tree, r) for r in rays)]
        yield ctx, torch.cuda.ExternalStream(ctx.stream), [torch.from_numpy(r).cuda() for r in rays], want


def _record(ctx, stream, launches):
    import torch

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for rays, out in launches:
            ctx.trace_closest_ptr(N, rays.data_ptr(), out.data_ptr())
    return graph


def test_replays_beside_queued_traces(setup):
    import torch

    ctx, stream, rays, want = setup
    out = [torch.zeros((N, 4), dtype=torch.int32, device="cuda") for _ in rays]
    graph = _record(ctx, stream, [(rays[0], out[0])])
    other = torch.cuda.Stream()
    for _ in range(4):
        for o in out:
            o.fill_(-7)
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            for _ in range(3):
                graph.replay()
        for _ in range(3):
            ctx.trace_closest_ptr(N, rays[1].data_ptr(), out[1].data_ptr())
        torch.cuda.synchronize()
        for o, w in zip(out, want):
            assert np.array_equal(o.cpu().numpy(), w)


def test_more_recorded_launches_than_counter_sets(setup):
    """Launches recorded after the counter sets are used up need none."""
    import torch

    ctx, stream, rays, want = setup
    out = torch.zeros((N, 4), dtype=torch.int32, device="cuda")
    first = _record(ctx, stream, [(rays[0], out)] * 130)
    last = _record(ctx, stream, [(rays[1], out)])
    for graph, w in ((last, want[1]), (first, want[0]), (last, want[1])):
        out.fill_(-7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), w)
        out.fill_(-7)
        torch.cuda.synchronize()
        ctx.trace_closest_ptr(N, rays[0].data_ptr(), out.data_ptr())
        ctx.synchronize()
        assert np.array_equal(out.cpu().numpy(), want[0])
