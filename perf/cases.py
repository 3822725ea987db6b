"""The work whose speed is followed on an MI355X: what users of this framework have it do, through its public entry
points (``pyapr.aprnet.cuda`` modules, ``apr_models.unet.APRUNet``), over the sizes, element types and directions that
occur.  Every APR is converted from a synthetic volume (``pyapr.synthetic``), the features are the particle intensities
(scaled and with noise by the seed) or N(0, 1), the networks are randomly initialised by the seed.

A case is a dict:
  kind      "layer"  one stencil convolution, forward          "layer_fb"  the same, forward and backward
            "chain"  convolution -> ReLU -> max pool -> upsample, forward and backward
            "infer"  APRUNet forward under no_grad             "train"     APRUNet forward, loss, backward
  volume    family of the synthetic volume (names of pyapr.synthetic.CONFIGS); z, x, y its size in pixels
  dtype     element type of the features (parameters are float32)
  cin, cout, ky (stencil 3x3x3: ky = 3; 1x5x5: ky = 5)         for the layers and the chain
  depth, norm ("fold": BatchNorm folded into the convolutions, "batch", "group"), batch    for the networks
"""
import functools
import math
import os
import sys

import torch

_PKG = os.path.abspath("apr-cnn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from apr_models.unet import APRUNet, fold_norms  # noqa: E402
from pyapr import APR, aprnet  # noqa: E402
from pyapr.aprnet import utils  # noqa: E402
from pyapr.converter import get_apr  # noqa: E402
from pyapr.synthetic import CONFIGS, pipeline_parameters, synth_volume  # noqa: E402

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # the smallest call: the first layer of a network on a 128^3 volume, where launches and latency count
        dict(name="first_layer_128", kind="layer", volume="spheres128", z=128, x=128, y=128, dtype="f32", cin=1, cout=16, ky=3),
        # a wide layer at full resolution, the layer the framework is quoted on (fp32, 23 M particles)
        dict(name="layer_32_f32", kind="layer", volume="blobs512", z=256, x=512, y=512, dtype="f32", cin=32, cout=32, ky=3),
        # a light-sheet-like volume, most tree nodes read by the convolution; odd sizes
        dict(name="layer_16_f32_sparse", kind="layer", volume="nuclei2048", z=255, x=1021, y=1000, dtype="f32", cin=16, cout=16, ky=3),
        # the operators of one encoder / decoder step, trained in fp32
        dict(name="chain_32_f32", kind="chain", volume="blobs512", z=192, x=384, y=384, dtype="f32", cin=32, cout=32, ky=3),
        # a wide 2-D layer of a large image, trained on bfloat16 features
        dict(name="wide_2d_bf16", kind="layer_fb", volume="spots16k", z=1, x=4096, y=4096, dtype="bf16", cin=64, cout=64, ky=5),
        # segmentation of a large volume: the largest case
        dict(name="infer_bf16_large", kind="infer", volume="nuclei1024", z=512, x=1024, y=512, dtype="bf16", depth=3, norm="fold", batch=1),
        # the same network on an ordinary volume in fp32
        dict(name="infer_f32", kind="infer", volume="blobs512", z=256, x=512, y=512, dtype="f32", depth=3, norm="fold", batch=1),
        # serving of small ragged tiles, one at a time
        dict(name="infer_bf16_tile", kind="infer", volume="blobs512", z=101, x=203, y=187, dtype="bf16", depth=3, norm="fold", batch=1),
        # inference with the class's default normalisation, which cannot be folded
        dict(name="infer_group_f32", kind="infer", volume="blobs512", z=128, x=256, y=256, dtype="f32", depth=3, norm="group", batch=1),
        # training on a batch of crops (the APRs of a batch differ in size)
        dict(name="train_f32_crops", kind="train", volume="blobs512", z=64, x=128, y=128, dtype="f32", depth=3, norm="group", batch=2),
        # training on a large crop with bfloat16 features
        dict(name="train_bf16", kind="train", volume="blobs512", z=160, x=320, y=319, dtype="bf16", depth=2, norm="batch", batch=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer_fb", "chain", "infer", "infer", "train"])
    # a bfloat16 training step of a small network amplifies the rounding of one layer through the others (a few per cent of
    # a gradient between two orders of summation): bfloat16 gradients are drawn layer by layer, and listed once whole
    dtype = "f32" if kind == "train" else rng.choice(["f32", "bf16"])
    if kind == "layer_fb" or (kind == "layer" and rng.random() < 0.2):                  # 2-D images
        cin, cout = rng.choice([16, 32, 64]), rng.choice([16, 32, 64])
        side = 4096 if dtype == "bf16" else 3000
        return dict(kind=kind, volume="spots16k", z=1, x=_log_int(rng, 400, side), y=_log_int(rng, 400, side), dtype=dtype, cin=cin,
                    cout=cout, ky=5)
    volume = rng.choice(["blobs512", "nuclei1024", "nuclei2048"])
    # side lengths of the volume: log-uniform volume, uneven edges
    most = {"layer": 400, "chain": 300, "infer": 620 if dtype == "bf16" else 380, "train": 250}[kind]
    side = math.exp(rng.uniform(math.log(72), math.log(most)))
    if volume == "nuclei1024":                # dense: four fifths of the pixels are particles
        side *= 0.8
    z, x, y = (max(40, int(side * rng.uniform(0.75, 1.2))) for _ in range(3))
    if kind in ("layer", "chain"):
        cin = rng.choice([1, 8, 16, 24, 32, 64]) if kind == "layer" else rng.choice([16, 24, 32])
        return dict(kind=kind, volume=volume, z=z, x=x, y=y, dtype=dtype, cin=cin, cout=rng.choice([16, 32, 48]), ky=3)
    if kind == "infer":
        return dict(kind=kind, volume=volume, z=z, x=x, y=y, dtype=dtype, depth=rng.choice([2, 3]), norm=rng.choice(["fold", "fold", "group"]),
                    batch=1)
    batch = rng.choice([1, 2, 3]) if side < 130 else 1
    return dict(kind=kind, volume=volume, z=z, x=x, y=y, dtype=dtype, depth=2, norm=rng.choice(["group", "batch"]), batch=batch)


# ------------------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=4)
def _volume(volume, z, x, y, b):
    """Access arrays and particle intensities of the b-th volume of a case; blob density of the family, whatever the size."""
    shape, blob, n, axes, amp, bg, iso, rel = CONFIGS[volume]
    blobs = max(1, round(n * z * x * y / math.prod(shape)))
    apr, parts = get_apr(synth_volume((z, x, y), 1000 + b, blob, blobs, axes, amp, bg, iso), params=pipeline_parameters(rel))
    return apr.get_state(), torch.from_numpy(parts)


def _volume_apr(case, b):
    """A new APR (no plan yet) and its particle intensities: the volumes of a case are the same for every seed, so that
    outputs have one shape; features, weights and gradients differ."""
    st, parts = _volume(case["volume"], case["z"], case["x"], case["y"], b)
    return APR.from_state(st[:3], *st[4:], parameters=st[3]), parts


def _network(case, gen):
    norm = "batch" if case["norm"] == "fold" else case["norm"]
    net = APRUNet(1, 3, depth=case["depth"], n_filters_base=16, n_stencils=2, norm=norm)
    with torch.no_grad():
        net.head.bias.copy_(0.1 * torch.randn(3, generator=gen))
        for m in net.modules():
            if getattr(m, "weight", None) is not None and m.weight.dim() == 6:           # He initialisation of the stencils
                m.weight.copy_(torch.randn(m.weight.shape, generator=gen) * (2.0 / math.prod(m.weight.shape[2:])) ** 0.5)
            if getattr(m, "running_mean", None) is not None:                             # statistics as training leaves them
                m.running_mean.copy_(0.1 * torch.randn(m.running_mean.shape, generator=gen))
                m.running_var.copy_(0.5 + torch.rand(m.running_var.shape, generator=gen))
    if case["kind"] == "train":
        return net.to(DEV).train()
    net = net.eval()
    return (fold_norms(net) if case["norm"] == "fold" else net).to(DEV)


def prepare(case, seed):
    dtype, gen = DTYPES[case["dtype"]], torch.Generator().manual_seed(seed)
    dgen = torch.Generator(device=DEV).manual_seed(seed)
    batch = case.get("batch", 1)
    aprs, parts = zip(*(_volume_apr(case, b) for b in range(batch)))
    aprs = list(aprs)
    for a in aprs:
        a.init_cuda()
    n = max(a.total_number_particles() for a in aprs)
    st = {"case": case, "aprs": aprs}
    if case["kind"] in ("infer", "train"):
        x = torch.zeros(batch, 1, n)
        for b, p in enumerate(parts):
            x[b, 0, :len(p)] = p * 1e-3
        # exposure and read-out noise of this acquisition
        x = x.to(DEV) * (0.8 + 0.4 * torch.rand(1, device=DEV, generator=dgen)) + 0.02 * torch.randn(x.shape, device=DEV, generator=dgen)
        st["x"] = x.to(dtype)
        st["net"] = _network(case, gen)
        if case["norm"] == "fold":
            st["net"].prepare_inference(aprs)
        if case["kind"] == "train":
            # three classes by intensity, one channel each (particles of a segmentation training set)
            cls = (st["x"].float() > 0.15).long() + (st["x"].float() > 0.6).long()
            st["target"] = torch.zeros(batch, 3, n, device=DEV).scatter_(1, cls, 1.0)
        return st
    cin, cout, k = case["cin"], case["cout"], (1, 5, 5) if case["ky"] == 5 else (3, 3, 3)
    st["conv"] = aprnet.cuda.APRConv(cin, cout, nstencils=2, kernel_size=k)
    with torch.no_grad():
        st["conv"].weight.copy_(torch.randn(st["conv"].weight.shape, generator=gen) * (1.0 / (cin * math.prod(k))) ** 0.5)
        st["conv"].bias.copy_(torch.randn(cout, generator=gen) * 0.1)
    st["conv"].to(DEV)
    st["x"] = torch.randn(1, cin, n, device=DEV, generator=dgen).to(dtype)
    if case["kind"] == "layer":
        return st
    st["x"].requires_grad_(True)
    if case["kind"] == "chain":
        st["pool"], st["up"] = aprnet.cuda.MaxPool(), aprnet.cuda.UpSampleConst()
    # a gradient of one sign and order of magnitude, as a loss over neighbouring particles sends it
    st["grad"] = (0.5 + torch.rand(1, cout, n, device=DEV, generator=dgen)).to(dtype)
    return st


# ---------------------------------------------------------------------------------------------------------- pass
def run(st):
    case, aprs, x = st["case"], st["aprs"], st["x"]
    kind = case["kind"]
    deltas = torch.zeros(len(aprs), dtype=torch.int32)
    if kind == "layer":
        with torch.no_grad():
            return st["conv"](x, aprs, deltas)
    if kind == "infer":
        with torch.no_grad():
            return st["net"](x, aprs)
    if kind == "train":
        net = st["net"]
        for p in net.parameters():
            p.grad = None
        logits = net(x, aprs)
        loss = torch.nn.functional.mse_loss(logits.float(), st["target"])
        loss.backward()
        return {"logits": logits.detach(), "loss": loss.detach(), "grads": [p.grad for p in net.parameters()],
                "statistics": [b for b in net.buffers() if b.dim() > 0]}
    conv = st["conv"]
    if kind == "layer_fb":
        y = conv(x, aprs, deltas)
    else:
        y = st["up"](st["pool"](torch.relu(conv(x, aprs, deltas)), aprs, deltas), aprs, deltas)
    return [y.detach(), *torch.autograd.grad(y, (x, conv.weight, conv.bias), st["grad"])]


# ---------------------------------------------------------------------------------------------------------- work
@functools.lru_cache(maxsize=None)
def _particles(volume, z, x, y, batch):
    """Feature counts per level delta 0..3 of the case's APRs."""
    aprs = [_volume_apr(dict(volume=volume, z=z, x=x, y=y), b)[0] for b in range(batch)]
    return [sum(utils.number_particles(a, d) for a in aprs) for d in range(4)]


def work(case):
    e = 2 if case["dtype"] == "bf16" else 4
    n = _particles(case["volume"], case["z"], case["x"], case["y"], case.get("batch", 1))
    if case["kind"] in ("layer", "layer_fb", "chain"):
        cin, cout, taps = case["cin"], case["cout"], 25 if case["ky"] == 5 else 27
        fwd = 2 * taps * cin * cout * n[0]
        access = 2 * n[0]                                  # y coordinate of every particle
        if case["kind"] == "layer":
            return {"bytes": e * (cin + cout) * n[0] + access, "flops": fwd}
        # backward: input gradient and weight gradient, the forward's products each; reads x and dY, writes y and dX
        return {"bytes": e * (2 * cin + 2 * cout) * n[0] + access, "flops": 3 * fwd}
    depth, widths = case["depth"], [16 * 2 ** i for i in range(4)]
    flops, backward_off = 0, 0
    cin = 1
    for i in range(depth + 1):                             # encoder: two convolutions per level
        flops += 2 * 27 * (cin * widths[i] + widths[i] ** 2) * n[i]
        cin = widths[i]
    for i in reversed(range(depth)):                       # decoder: 1x1x1, then two convolutions on the concatenation
        flops += 2 * widths[i + 1] * widths[i] * n[i + 1] + 2 * 27 * (2 * widths[i] ** 2 + widths[i] ** 2) * n[i]
    flops += 2 * widths[0] * 3 * n[0]
    if case["kind"] == "infer":
        return {"bytes": e * (1 + 3) * n[0] + 2 * n[0], "flops": flops}
    backward_off = 2 * 27 * widths[0] * n[0]               # the first layer needs no input gradient
    return {"bytes": e * (1 + 3) * n[0] + 4 * 3 * n[0] + 2 * n[0], "flops": 3 * flops - backward_off}


def tolerance(case):
    # Measured: fp32 against the same pass in 64 bits, bfloat16 against the fp32 matrix instructions on the same rounded
    # weights (another order of the fp32 sums before each rounding to bfloat16); about four times the largest seen is stated.
    f32 = case["dtype"] == "f32"
    kind = case["kind"]
    if kind == "layer":
        return {"rel": 3e-6, "max": 4e-5} if f32 else {"rel": 2e-4, "max": 0.03}
    if kind == "layer_fb":
        return {"rel": 1e-5, "max": 1e-4} if f32 else {"rel": 2e-4, "max": 0.03}
    if kind == "chain":                        # a pooled maximum that moves to its neighbour moves a whole gradient
        return {"rel": 3e-3, "max": 0.99}
    if kind == "infer":
        return {"rel": 1.5e-5, "max": 2e-4} if f32 else {"rel": 0.03, "max": 0.45}
    return {"rel": 5e-3, "max": 0.08} if f32 else {"rel": 0.03, "max": 0.6}
