"""The network's convolution and its weight gradient by themselves, on the
same bf16 operands as their references.

* The weight gradient is a sum in a stated order (1024 pixels at a time, one
  fp32 fmaf per pixel, then those sums in fp32): bit for bit against that
  sum in numpy.  Training depends on the order: Adam's first steps take the sign
  of a gradient, so another rounding of one that is about zero moves the
  weight the other way.  And a step is repeatable bit for bit.
* The convolution against 64 bits.  Its sums are in fp32, at most 9 x 224 + 63
  roundings of 2^-24 of a partial sum: a random walk of 2.7e-6 of the sum of
  the terms' magnitudes, and the tolerance is four of it.  One lost tap is
  1e-3 and more.
"""
import ctypes

import numpy as np
import pytest

from cvt_amd.net import ProposalNet

pytestmark = pytest.mark.gpu

CONV_TOL = 1.1e-5

# images of less than a matrix step, of a chunk and a remainder, of more
# chunks than one batch of the last addition; columns that a step skips; tiles
# of k with a half, with channels of both inputs, with an upsampled input; the
# head's 8 channels; every dilation
CASES = [
    # N, H, W, c1, c2, up2, cout, dil
    (1, 1, 1, 128, 0, 0, 128, 8),
    (3, 5, 1, 8, 0, 0, 32, 1),
    (3, 5, 7, 128, 0, 0, 128, 4),
    (1, 34, 65, 128, 0, 0, 128, 2),
    (2, 24, 44, 96, 128, 1, 96, 1),
    (1, 2, 6, 32, 64, 1, 32, 1),
    (1, 30, 70, 64, 48, 0, 96, 1),
    (1, 32, 96, 64, 0, 0, 64, 1),
    (5, 60, 64, 8, 0, 0, 32, 1),
    (3, 210, 216, 8, 0, 0, 8, 1),
    (2, 66, 130, 32, 0, 0, 8, 1),
]


def operands(N, H, W, c1, c2, up2, cout, dil, seed):
    import torch
    g = torch.Generator().manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).bfloat16()

    x1 = rnd(N, H, W, c1)
    x2 = None
    if c2:
        x2 = rnd(N, H // 2, W // 2, c2) if up2 else rnd(N, H, W, c2)
    cin = c1 + c2
    kpad, cpad = (9 * cin + 31) // 32 * 32, (cout + 31) // 32 * 32
    w = torch.zeros(cpad, kpad, dtype=torch.bfloat16)
    w[:cout, :9 * cin] = rnd(cout, 9 * cin)
    return x1, x2, w, rnd(N, H, W, cout)


def patches(x1, x2, up2, dil):
    """fp32 [pixel][k]: the taps of every pixel, zero beyond the image"""
    import torch
    x = x1.float()
    if x2 is not None:
        y = x2.float()
        if up2:
            y = y.repeat_interleave(2, 1).repeat_interleave(2, 2)
        x = torch.cat([x, y], -1)
    N, H, W, c = x.shape
    p = torch.nn.functional.pad(x, (0, 0, dil, dil, dil, dil))
    cols = [p[:, dy * dil:dy * dil + H, dx * dil:dx * dil + W]
            for dy in range(3) for dx in range(3)]
    return torch.stack(cols, 3).reshape(N * H * W, 9 * c).numpy()


def run(net, x1, x2, w, g, up2, dil, conv):
    import torch
    N, H, W, c1 = x1.shape
    cout = g.shape[3]
    dev = [t.cuda() if t is not None else None for t in (x1, x2, w, g)]
    y = torch.full((N, H, W, cout), float("nan"), device="cuda")
    dw = torch.zeros(w.shape, device="cuda")
    db = torch.zeros(w.shape[0], device="cuda")
    torch.cuda.synchronize()
    ptr = [ctypes.c_void_p(t.data_ptr() if t is not None else None)
           for t in dev + [y, dw, db]]
    net._check(net._lib.pm_net_conv_selftest(
        net.handle, ptr[0], c1, ptr[1], 0 if x2 is None else x2.shape[3],
        up2, N, H, W, cout, dil, ptr[2], ptr[4] if conv else None, ptr[3],
        ptr[5], ptr[6]))
    torch.cuda.synchronize()
    return y.cpu().numpy(), dw.cpu().numpy(), db.cpu().numpy()


@pytest.mark.parametrize("case", CASES)
def test_weight_gradient_is_the_sum_in_its_order(case):
    N, H, W, c1, c2, up2, cout, dil = case
    x1, x2, w, g = operands(*case, seed=H + W)
    x = patches(x1, x2, up2, dil)
    gv = g.float().reshape(-1, cout).numpy()
    sums = np.zeros((cout, x.shape[1]), np.float32)
    bias = np.zeros(cout, np.float32)
    for c in range(0, len(x), 1024):
        acc = np.zeros((cout, x.shape[1]), np.float32)
        accb = np.zeros(cout, np.float32)
        for p in range(c, min(c + 1024, len(x))):
            # a product of two bf16 is exact: this is one fmaf
            acc += np.multiply.outer(gv[p], x[p])
            accb += gv[p]
        sums += acc
        bias += accb
    with ProposalNet(seed=1) as net:
        _, dw, db = run(net, x1, x2, w, g, up2, dil, False)
    got = dw[:cout, :x.shape[1]]
    assert np.array_equal(got, sums), np.argwhere(got != sums)[:5]
    assert np.array_equal(db[:cout], bias)
    # the padding is left alone
    assert not dw[cout:].any() and not dw[:, x.shape[1]:].any()
    assert not db[cout:].any()


@pytest.mark.parametrize("case", CASES)
def test_convolution_against_64_bits(case):
    N, H, W, c1, c2, up2, cout, dil = case
    x1, x2, w, g = operands(*case, seed=H * W)
    x = patches(x1, x2, up2, dil).astype(np.float64)
    wk = w[:cout, :x.shape[1]].double().numpy().T
    with ProposalNet(seed=1) as net:
        y, _, _ = run(net, x1, x2, w, g, up2, dil, True)
    err = np.abs(y.reshape(-1, cout) - x @ wk)
    assert (err <= CONV_TOL * (np.abs(x) @ np.abs(wk))).all(), err.max()


def test_a_training_run_repeats_bit_for_bit():
    from cvt_amd import synth_gpu
    from test_gpu_net import batch
    x, t = batch(synth_gpu, 2, 88, 136, seed=5)
    got = []
    for _ in range(2):
        with ProposalNet(seed=9) as net:
            for _ in range(3):
                net.train_step(x.data_ptr(), t.data_ptr(), 2, 88, 136, 1e-3)
            got.append((net.grads(), net.params()))
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])
