"""pm_set_planes and a captured pm_iterate: a graph evaluates the planes that
are there when it is replayed, whatever their cost channel holds, and a
capture that is not replayed changes nothing.  At sizes of all three forms of
the propagate (teams, 64 x 4 tiles, wide tiles); every replay against the
eager calls, with eager work between the replays."""
import pytest

import cvt_amd
from test_gpu_parity import first_diff, same

pytestmark = pytest.mark.gpu

CENSUS, CG = cvt_amd.PM_COST_CENSUS, cvt_amd.PM_COST_COLOR_GRAD


def put(ctx, planes, iteration, cost):
    for v in (0, 1):
        q = planes[v].copy()
        q[..., 3] = cost
        ctx.set_planes(v, q, iteration)


def fields(ctx):
    return [ctx.planes(v) for v in (0, 1)]


@pytest.mark.parametrize("W,H,r", [(157, 83, 4), (400, 300, 1),
                                   (1100, 400, 3)])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_replay_on_a_callers_planes(synth, W, H, r, kind):
    import torch
    L, R, _ = synth.make_pair(W, H, cells=6, dmax=24.0, channels=4, seed=8)
    stream = torch.cuda.Stream()
    with cvt_amd.Context(radius=r, disparity_max=24.0, cost_kind=kind,
                         stream=stream.cuda_stream) as ctx:
        ctx.set_images(L, R)
        ctx.setup()
        ctx.iterate(1)
        mine = fields(ctx)
        ctx.setup()
        put(ctx, mine, 0, 0.5)
        ctx.iterate(2)
        want = fields(ctx)
        ctx.setup()
        ctx.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ctx.iterate(2)
        for cost in (0.0, 1.0, 1e30):
            ctx.setup()
            put(ctx, mine, 0, cost)
            ctx.sync()
            graph.replay()
            torch.cuda.synchronize()
            got = fields(ctx)
            for v in (0, 1):
                assert same(got[v], want[v]), (cost, v,
                                               first_diff(got[v], want[v]))
        del graph


@pytest.mark.parametrize("W,H,r", [(157, 83, 4), (1100, 400, 3)])
def test_a_capture_alone_does_not_cost_the_planes(synth, W, H, r):
    import torch
    L, R, _ = synth.make_pair(W, H, cells=6, dmax=24.0, channels=4, seed=9)
    stream = torch.cuda.Stream()
    with cvt_amd.Context(radius=r, disparity_max=24.0,
                         stream=stream.cuda_stream) as ctx:
        ctx.set_images(L, R)
        ctx.setup()
        ctx.iterate(1)
        mine = fields(ctx)
        ctx.setup()
        put(ctx, mine, 4, 0.0)
        ctx.iterate(1)
        want = fields(ctx)
        ctx.setup()
        put(ctx, mine, 2, 0.0)
        ctx.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ctx.iterate(2)
        assert ctx.iteration == 4
        ctx.iterate(1)
        got = fields(ctx)
        for v in (0, 1):
            assert same(got[v], want[v]), (v, first_diff(got[v], want[v]))
        del graph
