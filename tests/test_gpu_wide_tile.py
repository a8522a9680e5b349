"""The propagate's wide tiles (128 x 8 pixels with a window of the other
view in LDS, taken by images of at least 448 of them, 300 from a patch
radius of 4 on), the tame and the
general loops, and the costs it does not evaluate again, bit for bit
against the oracle or against the calls that evaluate them."""
import numpy as np
import pytest

import cvt_amd
from cvt_amd.batch import Batch
from test_gpu_parity import first_diff, same

pytestmark = pytest.mark.gpu

CENSUS, CG = cvt_amd.PM_COST_CENSUS, cvt_amd.PM_COST_COLOR_GRAD


def run(ctx, L, R, iters):
    ctx.set_images(L, R)
    ctx.setup()
    ctx.iterate(iters)
    return ctx.planes(0), ctx.planes(1)


def check(oracle, L, R, r, dmax, iters, kind, kw):
    want = oracle.run(L, R, r, dmax, iters, cost_kind=kind, cost_weight=kw)
    with cvt_amd.Context(radius=r, disparity_max=dmax, cost_kind=kind,
                         cost_weight=kw) as ctx:
        got = run(ctx, L, R, iters)
    assert same(got[0], want["stateL"]), first_diff(got[0], want["stateL"])
    assert same(got[1], want["stateR"]), first_diff(got[1], want["stateR"])


# partial tiles on both sides, a window wider than the image, windows of
# almost no range, two rows of very many tiles, the largest patch that fits
@pytest.mark.parametrize("W,H,C,r,dmax,iters,kind", [
    (2053, 219, 4, 3, 200.0, 1, CG),
    (1153, 263, 1, 5, 17.0, 2, CENSUS),
    (2049, 219, 4, 1, 3.5, 3, CENSUS),
    (28677, 9, 1, 2, 30.0, 2, CG),
    (1031, 275, 4, 8, 12.0, 1, CENSUS),
])
def test_wide_tiles_bitexact(oracle, synth, W, H, C, r, dmax, iters, kind):
    L, R, _ = synth.make_pair(W, H, cells=9, dmax=min(dmax, 60.0),
                              channels=C, seed=W)
    check(oracle, L, R, r, dmax, iters, kind, 25.5)


# values that leave the tame range: the general loops take the image
@pytest.mark.parametrize("value", [1e5, -1e-30, -0.0])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_untame_images_bitexact(oracle, synth, value, kind):
    L, R, _ = synth.make_pair(1030, 400, cells=9, dmax=30.0, channels=4,
                              seed=5)
    for img, x, y in ((L, 400, 100), (R, 611, 37)):
        img[y:y + 3, x:x + 4, 1] = value
    check(oracle, L, R, 2, 30.0, 2, kind, 16.0)


@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_iterating_in_one_call_and_in_several(synth, kind):
    """the flat proposal's cost, kept within a call, and the plane costs,
    kept from one iteration to the next"""
    L, R, _ = synth.make_pair(1100, 400, cells=9, dmax=30.0, channels=4,
                              seed=6)
    with cvt_amd.Context(radius=3, disparity_max=30.0, cost_kind=kind) as ctx:
        one = run(ctx, L, R, 3)
        ctx.setup()
        for _ in range(3):
            ctx.iterate(1)
        assert same(ctx.planes(0), one[0]) and same(ctx.planes(1), one[1])


@pytest.mark.parametrize("W,H", [(90, 40), (1100, 400)])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_a_callers_cost_channel_is_not_trusted(synth, W, H, kind):
    L, R, _ = synth.make_pair(W, H, cells=6, dmax=20.0, channels=4, seed=7)
    with cvt_amd.Context(radius=3, disparity_max=20.0, cost_kind=kind) as ctx:
        p = run(ctx, L, R, 1)
        ctx.iterate(2)
        want = ctx.planes(0), ctx.planes(1)
        for cost in (0.0, 1.0, 1e30):
            for v in (0, 1):
                q = p[v].copy()
                q[..., 3] = cost
                ctx.set_planes(v, q, 1)
            ctx.iterate(2)
            assert same(ctx.planes(0), want[0]), cost
            assert same(ctx.planes(1), want[1]), cost


@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_batch_of_wide_tiles_equals_single_pairs(synth, kind):
    import torch
    sizes = [(700, 301), (333, 517), (129, 9), (901, 240)]
    pairs, keep, want = [], [], []
    for i, (W, H) in enumerate(sizes):
        L, R, _ = synth.make_pair(W, H, cells=6, dmax=10.0 + 20 * i,
                                  channels=4, seed=40 + i)
        keep.append((torch.from_numpy(L).cuda(), torch.from_numpy(R).cuda()))
        pairs.append({"width": W, "height": H, "channels": 4,
                      "disparity_max": 10.0 + 20 * i,
                      "left": keep[i][0].data_ptr(),
                      "right": keep[i][1].data_ptr()})
        with cvt_amd.Context(radius=3, disparity_max=10.0 + 20 * i,
                             cost_kind=kind) as ctx:
            want.append(run(ctx, L, R, 3))
    torch.cuda.synchronize()
    with Batch(pairs, radius=3, cost_kind=kind) as b:
        for rows, wg in (None, 0), (8, 0), (8, 300), (4, 0):
            if rows:
                b.set_tuning(rows, wg)
            b.run(3)
            for i in range(len(sizes)):
                for v in (0, 1):
                    assert same(b.planes(i, v), want[i][v]), (rows, wg, i, v)
