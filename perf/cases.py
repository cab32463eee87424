"""The work this library is used for, as cases that can be timed and whose outputs can be compared.

Single layers are called as an application calls them (one call per layer on buffers it owns); chains of layers go
through the layer-table runner.  Sizes come from the benchmark's configurations and the test geometries."""
import json
import math

import numpy as np
import torch

from pulp_nn_amd import PulpNN, mobilenet, network

_LIBS = {}


def _lib(bits):
    """One loaded library per batch-norm width, on torch's current stream."""
    if bits not in _LIBS:
        _LIBS[bits] = PulpNN(bits)
    _LIBS[bits].use_torch_stream()
    return _LIBS[bits]


# ---- the cases ------------------------------------------------------------------------------------------------------

def listed():
    return [
        # one image of a small convolution: the latency of a single call
        dict(name="conv3x3_16x16_32to64_b1", kind="conv", bits=32, requant="bn", batch=1, h=16, w=16, ci=32, co=64, kx=3,
             ky=3, stride=1, pt=1, pb=1, pl=1, pr=1),
        # the same layer at the batch a throughput server runs
        dict(name="conv3x3_16x16_32to64_b256", kind="conv", bits=32, requant="bn", batch=256, h=16, w=16, ci=32, co=64, kx=3,
             ky=3, stride=1, pt=1, pb=1, pl=1, pr=1),
        # an early layer of a network with thin channels (24, 40: no multiples of 16) on an odd image, stride 2
        dict(name="conv3x3_s2_57x43_24to40_b32", kind="conv", bits=32, requant="mult", batch=32, h=57, w=43, ci=24, co=40,
             kx=3, ky=3, stride=2, pt=1, pb=1, pl=1, pr=1),
        # the large convolution: 64-bit batch-norm, padding on two sides only
        dict(name="conv3x3_64x64_256to256_bn64_b64", kind="conv", bits=64, requant="bn", batch=64, h=64, w=64, ci=256, co=256,
             kx=3, ky=3, stride=1, pt=1, pb=0, pl=1, pr=0),
        # the pointwise layer of the headline benchmark, scalar multiplier
        dict(name="pointwise_28x28_128to256_b256", kind="pointwise", bits=32, requant="mult", batch=256, h=28, w=28, ci=128,
             co=256),
        # depthwise layers: stride 1 on rows the application has padded, stride 2 through the generic entry point
        dict(name="depthwise3x3_s1_56x56x128_b256", kind="depthwise_s1", bits=32, requant="bn", batch=256, h=56, w=56, ch=128),
        dict(name="depthwise3x3_s2_56x56x128_b256", kind="depthwise", bits=32, requant="bn", batch=256, h=56, w=56, ch=128,
             kx=3, ky=3, stride=2, pt=1, pb=1, pl=1, pr=1),
        # a depthwise layer on odd planes with a channel tail
        dict(name="depthwise3x3_35x29x72_b32", kind="depthwise", bits=32, requant="bn", batch=32, h=35, w=29, ch=72, kx=3, ky=3,
             stride=1, pt=1, pb=1, pl=1, pr=1),
        # a classifier: 64 rows against a 4 MB weight matrix
        dict(name="linear_1024to4096_bn64_b64", kind="linear", bits=64, requant="bn", batch=64, k=1024, n=4096),
        # a whole network, one image (latency) and a full batch (throughput)
        dict(name="mobilenet_0.5_128_b1", kind="mobilenet", batch=1),
        dict(name="mobilenet_0.5_128_b256", kind="mobilenet", batch=256),
        # a residual block with everything around it: stem, max pooling, two convolutions, add, average pooling, linear
        dict(name="residual_32x32_c64_b64", kind="residual", bits=32, batch=64, size=32, c=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, lo, hi):
    """Half of them whole groups of 16, a third multiples of 8, the rest any number."""
    n, u = _log_int(rng, lo, hi), rng.random()
    step = 16 if u < 0.5 else 8 if u < 0.83 else 1
    return max(step, n // step * step) if n >= step else n


def draw(rng):
    kind = rng.choice(["conv", "conv", "pointwise", "pointwise", "depthwise", "depthwise", "depthwise_s1", "linear",
                       "mobilenet", "residual"])
    bits = rng.choice([32, 32, 64])
    batch = _log_int(rng, 1, 256)
    if kind == "mobilenet":
        return dict(kind=kind, batch=_log_int(rng, 2, 250))
    if kind == "residual":
        return dict(kind=kind, bits=bits, batch=batch, size=4 * rng.randint(4, 14), c=16 * rng.randint(3, 8))
    case = dict(kind=kind, bits=bits, requant=rng.choice(["bn", "bn", "mult"]), batch=batch)
    if kind == "linear":
        case.update(k=_channels(rng, 32, 4096), n=_channels(rng, 10, 4096))
        return case
    case.update(h=_log_int(rng, 7, 64), w=_log_int(rng, 7, 64))
    if kind == "conv":
        ci = _channels(rng, 3, 256)
        while ci in (16, 32):  # whole tiles of pixels only at these: the listed layers and the networks have them
            ci = _channels(rng, 3, 256)
        case.update(ci=ci, co=_channels(rng, 8, 256), kx=3, ky=3, stride=rng.choice([1, 1, 2]), pt=1, pb=1, pl=1, pr=1)
        if rng.random() < 0.15:
            case.update(kx=5, ky=5, pt=2, pb=2, pl=2, pr=2)
        elif rng.random() < 0.15:
            case.update(pb=0, pr=0)
    elif kind == "pointwise":
        case.update(ci=_channels(rng, 8, 512), co=_channels(rng, 8, 512))
    elif kind == "depthwise":
        case.update(ch=_channels(rng, 8, 512), kx=3, ky=3, stride=rng.choice([1, 2]), pt=1, pb=1, pl=1, pr=1)
        if rng.random() < 0.2:
            case.update(kx=5, ky=5, pt=2, pb=2, pl=2, pr=2)
    else:
        case.update(w=max(8, case["w"] // 2 * 2), ch=_channels(rng, 8, 512))
    # no larger than the listed ones of its kind
    most_bytes, most_flops = (206e6, 50e9)
    while case["batch"] > 1 and (work(case)["bytes"] > most_bytes or work(case)["flops"] > most_flops):
        case["batch"] = max(1, case["batch"] // 2)
    return case


# ---- sizes ----------------------------------------------------------------------------------------------------------

def _out_hw(c):
    if c["kind"] in ("pointwise", "depthwise_s1"):
        return c["h"], c["w"]
    return ((c["h"] + c["pt"] + c["pb"] - c["ky"]) // c["stride"] + 1,
            (c["w"] + c["pl"] + c["pr"] - c["kx"]) // c["stride"] + 1)


def _table_work(layers, in_shape, batch):
    """A chain: its input, its parameters and its result move once, what lies between need not leave the chip."""
    shapes = network.infer_shapes(layers, in_shape)
    macs = params = 0
    for L in layers:
        ho, wo, co = shapes[L["name"]]
        if "w" in L:
            params += L["w"].size + 9 * co
            macs += ho * wo * L["w"].size
    last = layers[-1]
    out = int(np.prod(shapes[last["name"]])) * (4 if last["op"] == "linear_out_32" else 1)
    return {"bytes": batch * (int(np.prod(in_shape)) + out) + params, "flops": 2 * batch * macs}


def work(case):
    c, b = case, case["batch"]
    if c["kind"] == "mobilenet":
        return _table_work(mobilenet.descriptor(_mobilenet(1)), (128, 128, 3), b)
    if c["kind"] == "residual":
        return _table_work(_residual(c, 0), (c["size"], c["size"], 3), b)
    per_channel = 1 + (2 * c["bits"] // 8 if c["requant"] == "bn" else 0)
    if c["kind"] == "linear":
        return {"bytes": b * (c["k"] + c["n"]) + c["n"] * (c["k"] + per_channel), "flops": 2 * b * c["k"] * c["n"]}
    ho, wo = _out_hw(c)
    if c["kind"] in ("conv", "pointwise"):
        taps = c["kx"] * c["ky"] if c["kind"] == "conv" else 1
        return {"bytes": b * (c["h"] * c["w"] * c["ci"] + ho * wo * c["co"]) + c["co"] * (taps * c["ci"] + per_channel),
                "flops": 2 * b * ho * wo * c["co"] * taps * c["ci"]}
    taps = 9 if c["kind"] == "depthwise_s1" else c["kx"] * c["ky"]
    rows = c["h"] + 2 if c["kind"] == "depthwise_s1" else c["h"]
    return {"bytes": b * c["ch"] * (rows * c["w"] + ho * wo) + c["ch"] * (taps + per_channel),
            "flops": 2 * b * ho * wo * c["ch"] * taps}


def tolerance(case):
    return "exact"  # integers throughout


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _shift(k_bytes, k_mean):
    """out_shift that spreads |acc * k| of uniform bytes over the output range (what calibration arrives at)."""
    sigma = 147.0 * 74.0 * math.sqrt(k_bytes) * k_mean
    return int(math.log2(4 * sigma)) - 7


def _seeded(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))

    def ints(lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int64 if dtype == torch.int64 else torch.int32
                             ).to(dtype)

    def small(lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=dtype)

    return (lambda shape: small(0, 256, shape, torch.uint8), lambda shape: small(-128, 128, shape, torch.int8), ints)


def _mobilenet(batch):
    """The chain with its seeded weights and the calibrated shifts; the input comes from the case's seed instead."""
    shifts = json.load(open(mobilenet.SHIFTS_FILE))["shifts"]
    return dict(mobilenet.build(1, shifts), batch=batch)


def _residual(c, seed):
    r = np.random.Generator(np.random.PCG64([seed, 1]))
    n, half = c["c"], c["size"] // 2

    def layer(k_bytes, co, shape, **more):
        lo, hi, lam, dt = (256, 1025, 2 ** 16, np.int32) if c["bits"] == 32 else (2 ** 20, 2 ** 24 + 1, 2 ** 36, np.int64)
        return dict(w=r.integers(-128, 128, size=shape, dtype=np.int8), bias=r.integers(-128, 128, size=co, dtype=np.int8),
                    k=r.integers(lo, hi, co).astype(dt), lam=r.integers(-lam, lam + 1, co).astype(dt), relu=1, bn=1, mult=0,
                    shift=_shift(k_bytes, (lo + hi) / 2), **more)

    same = dict(pads=(1, 1, 1, 1), strides=(1, 1))
    layers = [
        dict(layer(27, n, (n, 3, 3, 3), **same), op="conv", name="stem"),
        dict(op="maxpool", name="pool", kernel=(3, 3), strides=(2, 2), pads=(1, 1, 1, 1), out_hw=(half, half)),
        dict(layer(9 * n, n, (n, 3, 3, n), **same), op="conv", name="c1"),
        dict(layer(9 * n, n, (n, 3, 3, n), **same), op="conv", name="c2"),
        dict(op="add", name="sum", m1=1, m2=1, shift=1),
        dict(op="avgpool", name="gap", kernel=(4, 4), strides=(4, 4), out_hw=(half // 4, half // 4), lam=3, shift=5, add=5,
             requant=1),
        dict(layer(n * (half // 4) ** 2, 100, (100, n * (half // 4) ** 2)), op="linear", name="fc"),
    ]
    for L, src in zip(layers, ("input", "stem", "pool", "c1", ("c2", "pool"), "sum", "gap")):
        L["in"] = src
    return layers


def prepare(case, seed):
    c, b = case, case["batch"]
    u8, s8, ints = _seeded(seed)
    if c["kind"] == "mobilenet":
        return {"runner": mobilenet.Runner(_lib(32), _mobilenet(b)), "x": u8((b, 128, 128, 3))}
    if c["kind"] == "residual":
        shape = (c["size"], c["size"], 3)
        return {"runner": network.Runner(_lib(c["bits"]), _residual(c, seed), shape, b), "x": u8((b,) + shape)}
    nn = _lib(c["bits"])
    co = c.get("co", c.get("ch", c.get("n")))
    if c["requant"] == "bn":
        dt = torch.int32 if c["bits"] == 32 else torch.int64
        lo, hi, lim = (256, 1025, 2 ** 16) if c["bits"] == 32 else (2 ** 20, 2 ** 24 + 1, 2 ** 36)
        k, lam, mult, relu, bn, k_mean = ints(lo, hi, (co,), dt), ints(-lim, lim + 1, (co,), dt), 0, 1, 1, (lo + hi) / 2
    else:
        k, lam, mult, relu, bn, k_mean = None, None, 640, 1, 0, 640
    bias = s8((co,))
    if c["kind"] == "linear":
        x, w, out = u8((b, c["k"])), s8((co, c["k"])), torch.empty((b, co), dtype=torch.uint8, device="cuda")
        args = (x, bias, out, w, k, lam, mult, _shift(c["k"], k_mean), c["k"], co, relu, bn)
        return {"nn": nn, "batch": b, "call": nn.pulp_nn_linear, "args": args, "out": out}
    ho, wo = _out_hw(c)
    h, w_ = c["h"], c["w"]
    out = torch.empty((b, ho, wo, co), dtype=torch.uint8, device="cuda")
    if c["kind"] == "conv":
        x, w = u8((b, h, w_, c["ci"])), s8((co, c["ky"], c["kx"], c["ci"]))
        args = (x, None, bias, out, w, k, lam, mult, _shift(c["ky"] * c["kx"] * c["ci"], k_mean), w_, h, c["ci"], wo, ho, co,
                c["kx"], c["ky"], c["pt"], c["pb"], c["pl"], c["pr"], c["stride"], c["stride"], relu, bn)
        call = nn.pulp_nn_conv_Ho_parallel
    elif c["kind"] == "pointwise":
        x, w = u8((b, h, w_, c["ci"])), s8((co, 1, 1, c["ci"]))
        args = (x, None, bias, out, w, k, lam, mult, _shift(c["ci"], k_mean), w_, h, c["ci"], wo, ho, co, 1, 1, 0, 0, 0, 0, 1, 1,
                relu, bn)
        call = nn.pulp_nn_pointwise_HoWo_parallel
    elif c["kind"] == "depthwise":
        x, w = u8((b, co, h, w_)), s8((co, c["ky"], c["kx"]))
        args = (x, None, bias, out, w, None, k, lam, mult, _shift(c["ky"] * c["kx"], k_mean), w_, h, co, wo, ho, co, c["kx"],
                c["ky"], c["pt"], c["pb"], c["pl"], c["pr"], c["stride"], c["stride"], relu, bn)
        call = nn.pulp_nn_depthwise_generic
    else:
        x, w = u8((b, co, h + 2, w_)), s8((co, 3, 3))
        x[:, :, 0], x[:, :, -1] = 0, 0
        args = (x, out, h + 2, w_, co, 1, 1, w, _shift(9, k_mean), mult, k, lam, relu, bn)
        call = nn.pulp_nn_depthwise_3x3_s1
    return {"nn": nn, "batch": b, "call": call, "args": args, "out": out}


def run(state):
    if "runner" in state:
        return state["runner"].run(state["x"])
    state["nn"].set_batch(state["batch"])
    state["call"](*state["args"])
    return state["out"]
