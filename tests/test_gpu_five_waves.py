"""The propagate built for five wavefronts per SIMD, which batches and
red-black passes take where that saves a round of work-groups
(pm_engine.hip, saves_a_round): batches at 4 and at 2 tile rows against
single pairs, red-black against the oracle, right inside and right outside
its range."""
import pytest

import cvt_amd
from cvt_amd.batch import Batch
from test_gpu_parity import first_diff, same
from test_gpu_wide_tile import CENSUS, CG, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,r", [(CENSUS, 4), (CG, 2)])
@pytest.mark.parametrize("n", [10, 11, 14])   # 1000, 1100, 1400 of 64 x 4
def test_batches_equal_single_pairs(synth, kind, r, n):
    import torch
    W, H = 63, 397
    pairs, keep, want = [], [], []
    for i in range(2):
        L, R, _ = synth.make_pair(W, H, cells=6, dmax=9.0, channels=4,
                                  seed=70 + i)
        keep.append((torch.from_numpy(L).cuda(), torch.from_numpy(R).cuda()))
        with cvt_amd.Context(radius=r, disparity_max=9.0,
                             cost_kind=kind) as ctx:
            want.append(run(ctx, L, R, 2))
    pairs = [{"width": W, "height": H, "channels": 4, "disparity_max": 9.0,
              "left": keep[i % 2][0].data_ptr(),
              "right": keep[i % 2][1].data_ptr()} for i in range(n)]
    torch.cuda.synchronize()
    with Batch(pairs, radius=r, cost_kind=kind) as b:
        for rows in (4, 2):
            b.set_tuning(rows, 0)
            b.run(2)
            for i in range(n):
                for v in (0, 1):
                    assert same(b.planes(i, v), want[i % 2][v]), (rows, i, v)


@pytest.mark.parametrize("W,H", [(639, 845), (641, 845), (640, 1021)])
@pytest.mark.parametrize("kind", [CENSUS, CG])
def test_red_black_bitexact(oracle, synth, W, H, kind):
    L, R, _ = synth.make_pair(W, H, cells=9, dmax=20.0, channels=4, seed=W)
    sch = cvt_amd.PM_SCHEDULE_RED_BLACK
    want = oracle.run(L, R, 1, 20.0, 1, cost_kind=kind, cost_weight=25.5,
                      schedule=sch)
    with cvt_amd.Context(radius=1, disparity_max=20.0, cost_kind=kind,
                         cost_weight=25.5, schedule=sch) as ctx:
        got = run(ctx, L, R, 1)
    for v, name in enumerate(("stateL", "stateR")):
        assert same(got[v], want[name]), first_diff(got[v], want[name])
