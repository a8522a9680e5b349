"""The work the library is measured on: stereo pairs through the engine
(plain, PM-Huber, depthMap, learned), batches of pairs, and the proposal
network's forward pass and training step, each through its public entry
point, from the smallest gray pair to 1920 x 1080.

Sizes and options are those of bench.py, the tests, the training script and
the design notes.  Images come from the library's synthetic scene model
(Voronoi cells of slanted planes, Perlin texture, noise), made on the GPU
from a seed.
"""
import math

import numpy as np
import torch

import cvt_amd
from cvt_amd import net as net_mod
from cvt_amd import synth_gpu
from cvt_amd.batch import Batch

# FLOP per tap: census cost, colour+gradient cost, KLT step; per pixel and
# ROF step
_CENSUS_TAP, _COLOR_GRAD_TAP, _KLT_TAP, _ROF_PIXEL = 50, 59, 150, 100
_STREAM = None


def _stream():
    """The program's one stream, as bench.py has one for all its work."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM.cuda_stream


def listed():
    return [
        # one small gray pair with the default cost: the lowest latency a
        # caller sees
        {"name": "gray_320x240", "kind": "pair", "w": 320, "h": 240,
         "channels": 1, "radius": 5, "dmax": 32.0, "iterations": 3,
         "cost": "census", "schedule": "jacobi", "pp": "lrcheck"},
        # the drop-in class call on host images: PMHuberStereo.disparityMap
        # with its defaults (PM-Huber coupling, LR check)
        {"name": "disparity_map_640x480", "kind": "class_map", "w": 640,
         "h": 480, "channels": 4, "radius": 5, "dmax": 64.0,
         "iterations": 5, "map": "disparity"},
        # the class's depthMap on a driving-camera sized host pair, normals
        # included
        {"name": "depth_map_1242x375", "kind": "class_map", "w": 1242,
         "h": 375, "channels": 4, "radius": 4, "dmax": 128.0,
         "iterations": 8, "map": "depth"},
        # an odd-sized gray pair, large patch, red-black schedule, holes
        # filled
        {"name": "red_black_451x333", "kind": "pair", "w": 451, "h": 333,
         "channels": 1, "radius": 7, "dmax": 48.0, "iterations": 3,
         "cost": "color_grad", "schedule": "red_black", "pp": "fill"},
        # the benchmark's plain step
        {"name": "plain_1280x720", "kind": "pair", "w": 1280, "h": 720,
         "channels": 4, "radius": 4, "dmax": 128.0, "iterations": 8,
         "cost": "color_grad", "schedule": "jacobi", "pp": "lrcheck"},
        # the benchmark's learned step: left view seeded by the network,
        # one refine iteration
        {"name": "learned_1280x720", "kind": "learned", "w": 1280, "h": 720,
         "channels": 4, "radius": 4, "dmax": 128.0, "iterations": 1,
         "cost": "color_grad", "schedule": "jacobi", "pp": "lrcheck",
         "views": 1},
        # a full-HD pair with the reference's own cost: the largest
        {"name": "census_1920x1080", "kind": "pair", "w": 1920, "h": 1080,
         "channels": 4, "radius": 4, "dmax": 192.0, "iterations": 8,
         "cost": "census", "schedule": "jacobi", "pp": "lrcheck"},
        # uneven pairs in one graph launch
        {"name": "batch_16_pairs", "kind": "batch", "pairs": 16, "w": 960,
         "h": 540, "radius": 4, "iterations": 3, "cost": "color_grad",
         "learned": False},
        # the serving mix: uneven pairs, learned start, one refine iteration
        {"name": "serving_16_pairs", "kind": "batch", "pairs": 16, "w": 1920,
         "h": 1080, "radius": 4, "iterations": 1, "cost": "color_grad",
         "learned": True},
        # the network alone on a small frame and on the benchmark's
        {"name": "net_forward_320x240", "kind": "net_forward", "n": 1,
         "w": 320, "h": 240},
        {"name": "net_forward_1280x720", "kind": "net_forward", "n": 1,
         "w": 1280, "h": 720},
        # one step of the training script: forward, backward, Adam
        {"name": "train_step_8x512x384", "kind": "train", "n": 8, "w": 512,
         "h": 384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, odd sizes, 64 x 48 up to 1920 x 1080, and no
    more work than the largest listed one."""
    kind = rng.choice(["pair", "pair", "pair", "learned", "class_map",
                       "batch", "net_forward", "train"])
    w, h = _log_int(rng, 64, 1920), _log_int(rng, 48, 1080)
    if kind == "net_forward":
        return {"kind": kind, "n": rng.randint(1, 2), "w": (w + 7) // 8 * 8,
                "h": (h + 7) // 8 * 8}
    if kind == "train":
        return {"kind": kind, "n": rng.randint(1, 8),
                "w": min(w, 511) // 8 * 8, "h": min(h, 383) // 8 * 8}
    radius = rng.choice([2, 3, 4, 4, 5, 5, 7])
    iterations = rng.randint(1, 8)
    # at most the largest listed case's taps
    most = 81 * 8
    if kind == "class_map":
        radius, most = min(radius, 5), 81 * 6
    iterations = max(1, min(iterations, most // (2 * radius + 1) ** 2))
    if kind == "batch":
        radius = min(radius, 4)
    dmax = float(max(8, min(192, w // 10)))
    case = {"kind": kind, "w": w, "h": h, "radius": radius,
            "iterations": iterations}
    if kind == "batch":
        case.update(pairs=rng.randint(2, 16), iterations=min(iterations, 3),
                    cost=rng.choice(["census", "color_grad"]),
                    learned=rng.random() < 0.5, w=min(w, 960), h=min(h, 540))
        return case
    case.update(channels=rng.choice([1, 4, 4]), dmax=dmax)
    if kind == "class_map":
        case.update(map=rng.choice(["disparity", "depth"]))
        return case
    case.update(cost=rng.choice(["census", "color_grad"]),
                schedule=rng.choice(["jacobi", "jacobi", "jacobi",
                                     "red_black"]),
                pp=rng.choice(["none", "lrcheck", "fill"]))
    if case["schedule"] == "red_black" or case["cost"] == "color_grad":
        case["iterations"] = max(1, iterations // 2)
    if kind == "learned":
        case.update(views=rng.randint(1, 2),
                    iterations=min(case["iterations"], 2))
    return case


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------
def _images(w, h, channels, dmax, seed, n=1):
    """n pairs and their ground truth on the GPU."""
    left, right, gt = synth_gpu.make_pairs(n, w, h, cells=8, dmax=dmax,
                                           seed=seed)
    if channels == 1:
        left, right = (0.2126 * v[..., 0] + 0.7152 * v[..., 1] +
                       0.0722 * v[..., 2] for v in (left, right))
        left, right = left.contiguous(), right.contiguous()
    return left, right, gt


def _cost(name):
    return {"census": (cvt_amd.PM_COST_CENSUS, 16.0),
            "color_grad": (cvt_amd.PM_COST_COLOR_GRAD, 25.5)}[name]


def _pp(name):
    return {"none": cvt_amd.DISPARITY_PP_NONE,
            "lrcheck": cvt_amd.DISPARITY_PP_LRCHECK,
            "fill": cvt_amd.DISPARITY_PP_LRCHECK_FILL}[name]


def _pair_sizes(case, seed):
    """Uneven sizes of a batch: a third to all of the case's."""
    rng = np.random.default_rng(seed)
    sizes = []
    for _ in range(case["pairs"]):
        s = rng.uniform(1.0 / 3.0, 1.0)
        t = rng.uniform(0.85, 1.0)
        sizes.append((max(32, int(case["w"] * s)),
                      max(24, int(case["h"] * s * t))))
    return sizes


class _DeviceArray:
    """A batch's result where it lies in device memory, which is the
    batch's own: valid while the batch lives."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {
            "shape": shape, "typestr": "<f4", "data": (ptr, False),
            "version": 2, "strides": None}


def prepare(case, seed):
    kind = case["kind"]
    stream = _stream()
    if kind == "net_forward":
        left, right, _ = _images(case["w"], case["h"], 4, 96.0, seed,
                                 case["n"])
        x = torch.cat([left, right], -1).contiguous()
        out = torch.empty(case["n"], case["h"], case["w"], 4, device="cuda")
        net = net_mod.ProposalNet(stream=stream, weights=net_mod.WEIGHTS)
        torch.cuda.synchronize()
        return {"case": case, "x": x, "out": out, "net": net}
    if kind == "train":
        x, target = _training_batch(case, seed)
        net = net_mod.ProposalNet(stream=stream)
        net.set_params(_initial_weights(seed))
        torch.cuda.synchronize()
        return {"case": case, "x": x, "target": target, "net": net}
    if kind == "batch":
        keep, pairs = [], []
        # sizes are the case's, images the seed's
        for i, (w, h) in enumerate(_pair_sizes(case, 17)):
            dmax = max(8.0, 0.1 * w)
            left, right, _ = _images(w, h, 4, dmax, seed * 1009 + i)
            keep.append((left[0], right[0]))
            pairs.append({"width": w, "height": h, "channels": 4,
                          "disparity_max": dmax,
                          "left": keep[i][0].data_ptr(),
                          "right": keep[i][1].data_ptr()})
        ck, cw = _cost(case["cost"])
        torch.cuda.synchronize()
        net = None
        if case["learned"]:
            net = net_mod.ProposalNet(stream=stream, weights=net_mod.WEIGHTS)
        b = Batch(pairs, radius=case["radius"], cost_kind=ck, cost_weight=cw,
                  stream=stream)
        if net is not None:
            b.set_proposal(net, 1)
        there = [torch.as_tensor(_DeviceArray(b.disparity_ptr(i),
                                              b.shapes[i]), device="cuda")
                 for i in range(len(pairs))]
        out = [torch.empty(shape, device="cuda") for shape in b.shapes]
        torch.cuda.synchronize()
        return {"case": case, "batch": b, "net": net, "keep": keep,
                "there": there, "out": out}
    left, right, _ = _images(case["w"], case["h"], case["channels"],
                             case["dmax"], seed)
    left, right = left[0], right[0]
    if kind == "class_map":
        return {"case": case, "left": left.cpu().numpy(),
                "right": right.cpu().numpy(),
                "stereo": cvt_amd.PMHuberStereo()}
    ck, cw = _cost(case["cost"])
    ctx = cvt_amd.Context(
        radius=case["radius"], disparity_max=case["dmax"], stream=stream,
        cost_kind=ck, cost_weight=cw,
        schedule=(cvt_amd.PM_SCHEDULE_RED_BLACK
                  if case["schedule"] == "red_black"
                  else cvt_amd.PM_SCHEDULE_JACOBI))
    net = None
    if kind == "learned":
        net = net_mod.ProposalNet(stream=stream, weights=net_mod.WEIGHTS)
    out = torch.empty(case["h"], case["w"], device="cuda")
    torch.cuda.synchronize()
    return {"case": case, "left": left, "right": right, "ctx": ctx,
            "net": net, "out": out}


def _layout():
    """(weight offset, bias offset, floats of a padded weight row) of each
    convolution in the parameter vector."""
    off = 0
    for cin, cout, _ in net_mod.CONVS:
        kpad, cpad = -(-9 * cin // 32) * 32, -(-cout // 32) * 32
        woff = off
        off = -(-(off + cpad * kpad) // 64) * 64
        yield woff, off, kpad
        off = -(-(off + cpad) // 64) * 64


def _initial_weights(seed):
    """A network at the start of its training: He-normal weights, a small
    head with the mean disparity and a fronto-parallel normal as biases."""
    rng = np.random.default_rng(seed)
    w = np.zeros(net_mod.param_count(), np.float32)
    for k, ((cin, cout, _), (woff, boff, kpad)) in enumerate(
            zip(net_mod.CONVS, _layout())):
        head = k == len(net_mod.CONVS) - 1
        rows = w[woff:woff + cout * kpad].reshape(cout, kpad)
        rows[:, :9 * cin] = rng.standard_normal((cout, 9 * cin)) * (
            (2.0 / (9.0 * cin)) ** 0.5 * (0.1 if head else 1.0))
        if head:
            w[boff] = 0.35
            w[boff + 3] = 1.0
    return w


def _training_batch(case, seed):
    """Input pairs and plane targets (disparity / 128 and normal; no target
    in a thin band along the image border, where a left-right check rejects
    pixels)."""
    left, right, gt = _images(case["w"], case["h"], 4, 96.0, seed, case["n"])
    x = torch.cat([left, right], -1).contiguous()
    dx = torch.diff(gt, dim=2, append=gt[:, :, -1:]).clamp(-0.2, 0.2)
    dy = torch.diff(gt, dim=1, append=gt[:, -1:]).clamp(-0.2, 0.2)
    nz = 1.0 / torch.sqrt(dx * dx + dy * dy + 1.0)
    d = gt / 128.0
    d[:, :, :8] = -1.0
    target = torch.stack([d, -dx * nz, -dy * nz, nz], -1).contiguous()
    return x, target


# ---------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "net_forward":
        state["net"].forward(state["x"].data_ptr(), case["n"], case["h"],
                             case["w"], state["out"].data_ptr())
        return {"out": state["out"]}
    if kind == "train":
        # the learning rate of the end of the script's decay
        loss = state["net"].train_step(
            state["x"].data_ptr(), state["target"].data_ptr(), case["n"],
            case["h"], case["w"], 5e-5)
        return {"loss": loss, "grads": state["net"].grads()}
    if kind == "batch":
        # the program takes the results into tensors of its own
        state["batch"].run(case["iterations"])
        with torch.cuda.stream(_STREAM):
            for mine, there in zip(state["out"], state["there"]):
                mine.copy_(there)
        return state["out"]
    if kind == "class_map":
        s = state["stereo"]
        if case["map"] == "depth":
            d, n = s.depthMap(state["left"], state["right"], case["radius"],
                              case["dmax"], case["iterations"],
                              normalmap=True)
            return {"depth": d, "normals": n}
        return {"disparity": s.disparityMap(
            state["left"], state["right"], case["radius"], case["dmax"],
            case["iterations"])}
    ctx = state["ctx"]
    ctx.set_images_device(state["left"].data_ptr(), state["right"].data_ptr(),
                          case["w"], case["h"], case["channels"])
    if kind == "learned":
        ctx.setup_proposal(state["net"], case["views"])
    else:
        ctx.setup()
    ctx.iterate(case["iterations"])
    ctx.disparity_device(state["out"].data_ptr(), _pp(case["pp"]))
    return {"disparity": state["out"]}


# ---------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------
def _engine_flops(w, h, radius, iterations, census):
    """Both views' iterations: 10 cost evaluations and 6 KLT passes of a
    patch per pixel."""
    taps = (2 * radius + 1) ** 2
    tap = _CENSUS_TAP if census else _COLOR_GRAD_TAP
    return 2.0 * w * h * iterations * taps * (10 * tap + 6 * _KLT_TAP)


def work(case):
    kind = case["kind"]
    if kind == "net_forward":
        return {"bytes": 4.0 * case["n"] * case["h"] * case["w"] * 12 +
                4.0 * net_mod.param_count(),
                "flops": net_mod.forward_flops(case["h"], case["w"],
                                               case["n"])}
    if kind == "train":
        # forward, the weights' gradient and the input's; the parameters,
        # their gradient and the two moments read and written
        return {"bytes": 4.0 * case["n"] * case["h"] * case["w"] * 12 +
                4.0 * 8 * net_mod.param_count(),
                "flops": 3.0 * net_mod.forward_flops(case["h"], case["w"],
                                                     case["n"])}
    if kind == "batch":
        sizes = _pair_sizes(case, 17)
        flops = sum(_engine_flops(w, h, case["radius"], case["iterations"],
                                  case["cost"] == "census")
                    for w, h in sizes)
        if case["learned"]:
            flops += sum(net_mod.forward_flops(h, w) for w, h in sizes)
        return {"bytes": sum(4.0 * w * h * 9 for w, h in sizes),
                "flops": flops}
    w, h = case["w"], case["h"]
    n = case["iterations"]
    if kind == "class_map":
        if case["map"] == "disparity":
            n |= 1
        flops = _engine_flops(w, h, case["radius"], n, True) + \
            2.0 * w * h * n * 40 * _ROF_PIXEL
        return {"bytes": 4.0 * w * h * (2 * case["channels"] +
                                        (5 if case["map"] == "depth" else 1)),
                "flops": flops}
    flops = _engine_flops(w, h, case["radius"], n, case["cost"] == "census")
    if kind == "learned":
        flops += net_mod.forward_flops(h, w, case["views"])
    return {"bytes": 4.0 * w * h * (2 * case["channels"] + 1),
            "flops": flops}


# ---------------------------------------------------------------------
# the network in 64 bits
# ---------------------------------------------------------------------
def _parameters(vector):
    """Per convolution its weight (3, 3, cin, cout) and bias, in 64 bits."""
    w = torch.from_numpy(vector).double().cuda()
    got = []
    for (cin, cout, _), (woff, boff, kpad) in zip(net_mod.CONVS, _layout()):
        rows = w[woff:woff + cout * kpad].view(cout, kpad)[:, :9 * cin]
        weight = rows.reshape(cout, 3, 3, cin).permute(1, 2, 3, 0)
        got.append((weight.contiguous().requires_grad_(),
                    w[boff:boff + cout].clone().requires_grad_()))
    return got


def _conv(x, weight, bias, dil=1, relu=True):
    n, h, w, c = x.shape
    p = torch.nn.functional.pad(x, (0, 0, dil, dil, dil, dil))
    out = bias
    for ky in range(3):
        for kx in range(3):
            s = p[:, ky * dil:ky * dil + h, kx * dil:kx * dil + w]
            out = out + (s.reshape(-1, c) @ weight[ky, kx]).view(n, h, w, -1)
    return out.clamp_min(0.0) if relu else out


def _box(x, k):
    n, h, w, c = x.shape
    return x.view(n, h // k, k, w // k, k, c).mean((2, 4))


def _up(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2)


def _cost_volume(x, levels):
    n, h, w, _ = x.shape
    a, b = x[..., :3], x[..., 4:7]
    ys = torch.arange(h, device=x.device)
    xs = torch.arange(w, device=x.device)
    out = []
    for d in range(levels):
        s = 0.0
        for j in (-1, 0, 1):
            yy = (ys + j).clamp(0, h - 1)
            for i in (-1, 0, 1):
                xa, xb = (xs + i).clamp(0, w - 1), (xs + i - d).clamp(0, w - 1)
                s = s + (a[:, yy][:, :, xa] - b[:, yy][:, :, xb]).abs().sum(-1)
        out.append(s / 9.0)
    return torch.stack(out, -1)


def _network(x, params):
    it = iter(params)

    def conv(v, dil=1, relu=True):
        weight, bias = next(it)
        return _conv(v, weight, bias, dil, relu)

    cv = _cost_volume(_box(x, 4), 48)
    cv1 = _cost_volume(_box(x, 2), 64)
    e0 = conv(conv(x))
    e1 = conv(conv(torch.cat([_box(e0, 2), cv1], -1)))
    e2 = conv(conv(torch.cat([_box(e1, 2), cv], -1)))
    b = conv(conv(conv(conv(_box(e2, 2)), 2), 4), 8)
    d2 = conv(conv(torch.cat([e2, _up(b)], -1)))
    d1 = conv(conv(torch.cat([e1, _up(d2)], -1)))
    d0 = conv(conv(torch.cat([e0, _up(d1)], -1)))
    return conv(d0, relu=False)


def exact(case, seed):
    """The network's outputs in 64 bits.  The engine's planes have no such
    value: a plane is the survivor of comparisons, which another rounding
    decides otherwise."""
    if case["kind"] == "net_forward":
        left, right, _ = _images(case["w"], case["h"], 4, 96.0, seed,
                                 case["n"])
        x = torch.cat([left, right], -1).double()
        params = _parameters(net_mod.read_weights(net_mod.WEIGHTS))
        with torch.no_grad():
            return {"out": torch.cat([_network(x[i:i + 1], params)
                                      for i in range(case["n"])])}
    if case["kind"] == "train":
        x, target = _training_batch(case, seed)
        x, target = x.double(), target.double()
        params = _parameters(_initial_weights(seed))
        wn = torch.tensor([1.0, 0.05, 0.05, 0.05], device="cuda",
                          dtype=torch.float64)
        npix = case["n"] * case["h"] * case["w"]
        loss = 0.0
        for i in range(case["n"]):
            valid = (target[i:i + 1, ..., :1] >= 0.0).double()
            part = ((_network(x[i:i + 1], params) - target[i:i + 1]).abs() *
                    wn * valid).sum() / npix
            part.backward()
            loss += float(part.detach())
        grads = torch.zeros(net_mod.param_count(), dtype=torch.float64)
        for (weight, bias), (cin, cout, _), (woff, boff, kpad) in zip(
                params, net_mod.CONVS, _layout()):
            g = weight.grad.permute(3, 0, 1, 2).reshape(cout, 9 * cin).cpu()
            rows = grads[woff:woff + cout * kpad].view(cout, kpad)
            rows[:, :9 * cin] = g
            grads[boff:boff + cout] = bias.grad.cpu()
        return {"loss": loss, "grads": grads}
    return None
