"""The matrix-core weight gradient at the edges of its 64 x 4 pixel tiles:
images smaller than a tile, partial tiles in both directions at every level
and dilation, more than one tile per image and several images, against
torch autograd of the same network (test_gpu_net.py's reference and
tolerance)."""
import numpy as np
import pytest

from test_gpu_net import (GRAD_RTOL, batch, layout, ref_forward, ref_loss,
                          torch_weights)

from cvt_amd.net import ProposalNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W", [(1, 8, 8), (3, 40, 72), (2, 24, 136),
                                   (1, 72, 528)])
def test_gradients_at_tile_edges(N, H, W):
    from cvt_amd import synth_gpu
    x, t = batch(synth_gpu, N, H, W, seed=H + W)
    with ProposalNet(seed=23) as net:
        params = net.params()
        net.train_step(x.data_ptr(), t.data_ptr(), N, H, W, 1e-6, 1.0, 0.05)
        g = net.grads()
    ws = [(w.clone().requires_grad_(), b.clone().requires_grad_())
          for w, b in torch_weights(params)]
    o = ref_forward(x.cpu().permute(0, 3, 1, 2).contiguous(), ws)
    ref_loss(o, t.cpu().permute(0, 3, 1, 2), 1.0, 0.05).backward()
    for l, ((w, b), (woff, boff, cin, cout, kpad, cpad)) in \
            enumerate(zip(ws, layout()[0])):
        rows = g[woff:woff + cpad * kpad].reshape(cpad, kpad)
        got = rows[:cout, :9 * cin].reshape(cout, 3, 3, cin)
        want = w.grad.numpy().transpose(0, 2, 3, 1)
        n = 4 if cout == 8 else cout      # the head: 4 real outputs
        err = np.linalg.norm(got[:n] - want[:n]) / \
            max(np.linalg.norm(want[:n]), 1e-12)
        assert err < GRAD_RTOL, (l, err)
        gb, rb = g[boff:boff + n], b.grad.numpy()[:n]
        err = np.linalg.norm(gb - rb) / max(np.linalg.norm(rb), 1e-12)
        assert err < GRAD_RTOL, (l, "bias", err)
        # the padding of the rows and the unused rows stay zero
        assert not rows[:, 9 * cin:].any() and not rows[cout:].any(), l
