"""The propagate's teams of four lanes per pixel, which small images take
(patch taps that four divides with a remainder of 1 and of 3, fewer taps than
lanes, partial tiles, images smaller than a patch, both schedules, tame and
untame images), and the one-lane tiles right above their line, bit for bit
against the oracle."""
import pytest

import cvt_amd
from test_gpu_parity import first_diff, same

pytestmark = pytest.mark.gpu

CENSUS, CG = cvt_amd.PM_COST_CENSUS, cvt_amd.PM_COST_COLOR_GRAD


@pytest.mark.parametrize("W,H,C,r,dmax,iters,red_black,value", [
    (17, 5, 1, 1, 6.0, 3, False, None),
    (61, 33, 4, 2, 14.0, 2, True, None),
    (79, 21, 1, 3, 16.0, 2, False, None),
    (97, 31, 4, 8, 12.0, 1, True, None),
    (9, 7, 4, 10, 5.0, 2, False, None),
    (50, 30, 4, 2, 12.0, 2, False, 1e5),
    (50, 30, 4, 3, 12.0, 2, True, -0.0),
    (375, 300, 1, 1, 30.0, 1, False, None),    # the last of the teams
    (376, 300, 1, 1, 30.0, 1, False, None),    # one lane per pixel
    (376, 300, 4, 1, 30.0, 1, True, None),
])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_teams_bitexact(oracle, synth, W, H, C, r, dmax, iters, red_black,
                        value, kind):
    L, R, _ = synth.make_pair(W, H, cells=5, dmax=dmax, channels=C, seed=W)
    if value is not None:
        L[11:14, 20:24, 1] = value
        R[7:9, 31:33, 0] = value
    schedule = (cvt_amd.PM_SCHEDULE_RED_BLACK if red_black
                else cvt_amd.PM_SCHEDULE_JACOBI)
    want = oracle.run(L, R, r, dmax, iters, cost_kind=kind, cost_weight=25.5,
                      schedule=schedule)
    with cvt_amd.Context(radius=r, disparity_max=dmax, cost_kind=kind,
                         cost_weight=25.5, schedule=schedule) as ctx:
        ctx.set_images(L, R)
        ctx.setup()
        ctx.iterate(iters)
        for view, name in enumerate(("stateL", "stateR")):
            got = ctx.planes(view)
            assert same(got, want[name]), first_diff(got, want[name])
