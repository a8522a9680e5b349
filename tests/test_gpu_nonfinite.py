"""Images with infinities and NaN in the propagate's wide tiles and teams,
against the counted call, which takes the general loops of the 64 x 4 tiles.
(Not against the oracle: the cost reads gradients' sign bits, and the CPU's
NaN has another.)"""
import pytest

import cvt_amd
from test_gpu_parity import first_diff, same
from test_gpu_wide_tile import CENSUS, CG, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,r", [(1100, 400, 2), (161, 83, 3)])
@pytest.mark.parametrize("value", ["inf", "-inf", "nan"])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_images_that_are_not_finite(synth, W, H, r, value, kind):
    L, R, _ = synth.make_pair(W, H, cells=9, dmax=30.0, channels=4, seed=5)
    for img, x, y in ((L, W // 3, H // 4), (R, W // 2, H // 9)):
        img[y:y + 3, x:x + 4, 1] = float(value)
    with cvt_amd.Context(radius=r, disparity_max=30.0,
                         cost_kind=kind) as ctx:
        got = run(ctx, L, R, 2)
        ctx.setup()
        ctx.iterate_counted(2)
        for v in (0, 1):
            want = ctx.planes(v)
            assert same(got[v], want), first_diff(got[v], want)
