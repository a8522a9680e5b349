"""The convolution kernels at the edges of their tiles: images smaller than
a tile, partial tiles at every level and dilation, fewer and more tiles than
the walking kernel has work-groups, both tiles of the lattice kernel, and an
output that is not aligned for vector stores (the network's forward pass
against test_gpu_net.py's reference and tolerance)."""
import numpy as np
import pytest

from test_gpu_net import FWD_RTOL, batch, ref_forward, torch_weights

from cvt_amd.net import ProposalNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W", [(1, 8, 8), (2, 40, 56), (3, 24, 136),
                                   (1, 520, 528)])
def test_forward_at_tile_edges(N, H, W):
    import torch
    from cvt_amd import synth_gpu
    x, _ = batch(synth_gpu, N, H, W, seed=H + W)
    room = torch.full((N * H * W * 4 + 4,), float("nan"), device="cuda")
    got = []
    with ProposalNet(seed=29) as net:
        params = net.params()
        for skip in (0, 1):               # floats before the output
            torch.cuda.synchronize()
            net.forward(x.data_ptr(), N, H, W, room.data_ptr() + 4 * skip)
            torch.cuda.synchronize()
            got.append(room[skip:skip + N * H * W * 4].cpu().numpy().copy())
    want = ref_forward(x.cpu().permute(0, 3, 1, 2).contiguous(),
                       torch_weights(params))[:, :4]
    want = want.permute(0, 2, 3, 1).numpy().reshape(-1)
    assert np.linalg.norm(got[0] - want) < FWD_RTOL * np.linalg.norm(want)
    assert np.array_equal(got[0], got[1])
    assert torch.isnan(room[N * H * W * 4 + 1:]).all()  # nothing beyond
