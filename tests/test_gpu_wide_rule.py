"""Which images take the propagate's wide tiles: enough of them, little more
padding than with 64 x 4 tiles (pm_engine.hip, wide_pays), and a window that
fits a CU's LDS.  Both sides of every line, bit for bit against the oracle,
and batches against single pairs."""
import pytest

import cvt_amd
from cvt_amd.batch import Batch
from test_gpu_parity import same
from test_gpu_wide_tile import CENSUS, CG, check, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,C,r,dmax,iters,kind", [
    # the last tile column has one pixel in its first or in its second half
    (2113, 219, 4, 3, 200.0, 1, CG),
    (2113, 223, 1, 1, 3.5, 3, CENSUS),
    (28737, 16, 1, 2, 30.0, 1, CG),
    (1217, 263, 1, 5, 17.0, 2, CENSUS),
    (1153, 359, 4, 4, 60.0, 1, CG),
    # half a tile column too much below 448 tiles; below radius 4
    (1153, 263, 4, 4, 17.0, 1, CENSUS),
    (1153, 399, 4, 2, 17.0, 1, CG),
    # the largest windows that fit a CU, and the first that does not
    (1100, 276, 4, 9, 12.0, 1, CENSUS),
    (1100, 276, 4, 10, 12.0, 1, CENSUS),
    (1100, 276, 4, 11, 12.0, 1, CENSUS),
    # narrow images, as teams or as 64 x 4 tiles
    (258, 800, 4, 5, 25.0, 1, CENSUS),
    (130, 2400, 4, 4, 12.0, 1, CG),
    (16, 2400, 1, 3, 5.0, 1, CENSUS),
])
def test_both_sides_bitexact(oracle, synth, W, H, C, r, dmax, iters, kind):
    L, R, _ = synth.make_pair(W, H, cells=9, dmax=min(dmax, 60.0),
                              channels=C, seed=W + r)
    check(oracle, L, R, r, dmax, iters, kind, 25.5)


@pytest.mark.parametrize("kind", [CENSUS, CG])
@pytest.mark.parametrize("sizes", [
    [(700, 301), (333, 517), (129, 9), (901, 240)],    # wide tiles
    [(140, 200)] * 16,                                 # too much padding
])
def test_batches_equal_single_pairs(synth, sizes, kind):
    import torch
    pairs, keep, want = [], [], []
    for i, (W, H) in enumerate(sizes):
        L, R, _ = synth.make_pair(W, H, cells=6, dmax=10.0 + 2 * i,
                                  channels=4, seed=40 + i)
        keep.append((torch.from_numpy(L).cuda(), torch.from_numpy(R).cuda()))
        pairs.append({"width": W, "height": H, "channels": 4,
                      "disparity_max": 10.0 + 2 * i,
                      "left": keep[i][0].data_ptr(),
                      "right": keep[i][1].data_ptr()})
        with cvt_amd.Context(radius=4, disparity_max=10.0 + 2 * i,
                             cost_kind=kind) as ctx:
            want.append(run(ctx, L, R, 2))
    torch.cuda.synchronize()
    with Batch(pairs, radius=4, cost_kind=kind) as b:
        for rows, wg in (None, 0), (8, 0), (8, 300), (4, 0):
            if rows:
                b.set_tuning(rows, wg)
            b.run(2)
            for i in range(len(sizes)):
                for v in (0, 1):
                    assert same(b.planes(i, v), want[i][v]), (rows, wg, i, v)
