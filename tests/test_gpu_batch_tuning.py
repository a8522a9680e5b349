"""The shape that a batch reports is the one it runs: setting it again changes
nothing, wide or not, and keeps the last run's results."""
import pytest

from cvt_amd.batch import Batch
from test_gpu_parity import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,rows", [(640, 360, 8), (120, 90, 4)])
def test_setting_the_reported_shape_changes_nothing(synth, W, H, rows):
    import torch
    keep, pairs = [], []
    for i in range(2):
        L, R, _ = synth.make_pair(W, H, cells=6, dmax=12.0, channels=4,
                                  seed=60 + i)
        keep.append((torch.from_numpy(L).cuda(), torch.from_numpy(R).cuda()))
        pairs.append({"width": W, "height": H, "channels": 4,
                      "disparity_max": 12.0,
                      "left": keep[i][0].data_ptr(),
                      "right": keep[i][1].data_ptr()})
    torch.cuda.synchronize()
    with Batch(pairs, radius=4) as b:
        t = b.tuning
        assert (t["tile_rows"], t["workgroups"]) == (rows, 0)
        b.run(2)
        want = [b.planes(i, v) for i in range(2) for v in (0, 1)]
        b.set_tuning(t["tile_rows"], t["workgroups"])
        got = [b.planes(i, v) for i in range(2) for v in (0, 1)]
        assert all(same(g, w) for g, w in zip(got, want))
        assert b.tuning == t
        # and a tuned shape is the one that is timed and then runs
        table = b.autotune(reps=1)
        best = min(table, key=lambda c: c["ms"])
        assert b.tuning["tile_rows"] == best["tile_rows"]
        b.run(2)
        got = [b.planes(i, v) for i in range(2) for v in (0, 1)]
        assert all(same(g, w) for g, w in zip(got, want))
