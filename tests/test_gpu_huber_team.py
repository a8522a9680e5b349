"""Teams of four lanes per pixel beside PM-Huber smoothing, right below and
right above their line there (pm_engine.hip, team_pays), where radius 5 takes
the propagate built for five wavefronts and radius 1 the one for four, bit for
bit against the oracle."""
import pytest

import cvt_amd
from test_gpu_huber import assert_same, huber_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,r,n", [
    (250, 270, 1, 2), (251, 270, 1, 2),     # 90000 slots per tap
    (387, 388, 5, 1), (388, 388, 5, 1),     # 163840
])
def test_both_sides_of_the_line(oracle, synth, W, H, r, n):
    L, R, _ = synth.make_pair(W, H, cells=5, dmax=20.0, channels=4, seed=W)
    ref = oracle.run_huber(L, R, r, 20.0, n, 1e-4, 1.0, 5.0)
    with huber_ctx(r, 20.0, theta_min=1e-4) as ctx:
        ctx.set_images(L, R)
        ctx.setup()
        ctx.iterate(n)
        got = {"stateL": ctx.planes(0), "stateR": ctx.planes(1),
               "smoothL": ctx.smooth(0), "smoothR": ctx.smooth(1),
               "disp": ctx.disparity(cvt_amd.DISPARITY_PP_LRCHECK, 1.0, 5.0)}
    for k, v in got.items():
        assert_same(v, ref[k], k)
