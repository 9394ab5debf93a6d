"""Performance cases: the work that a program built on armnn_amd has the device do, through the public entry points.

A case is one of four kinds:
  network    a whole quantized classifier (armnn_amd.nets) through armnn_amd.executor.DeviceNetwork, configured as bench.py
             configures it (recommended fusions on, the captured pass replayed, two lanes for wide batches of a network
             without depthwise layers).  io "device": the images are already in HBM and the results stay there
             (DeviceNetwork.enqueue); io "host": images come from and results go to ordinary host arrays
             (DeviceNetwork.run).
  conv       one Convolution2d plan (shim.Conv2dPlan.run) on tensors resident in HBM, with a fused ReLU6
  depthwise  one DepthwiseConvolution2d plan, likewise
  fc         one FullyConnected plan (shim.FullyConnectedPlan.run), likewise

listed() holds the cases that are always measured, draw() gives further ones of the same ranges.  All outputs are 8-bit
codes computed with exact integer accumulation and the reference's own rounding, so results are compared exactly.
"""
import functools
import math

import numpy as np
import torch

from armnn_amd import nets, shim, synth
from armnn_amd.executor import DeviceNetwork
from armnn_amd.tensor import DataType, QTensor, TensorInfo


def _network(name, net, batch, resolution=224, width=1.0, weights="per_channel_s8", io="device"):
    return dict(name=name, kind="network", net=net, batch=batch, resolution=resolution, width=width, weights=weights, io=io)


def _conv(name, batch, h, w, ci, co, k, stride, u8):
    return dict(name=name, kind="conv", batch=batch, h=h, w=w, ci=ci, co=co, k=k, stride=stride, u8=u8)


def _depthwise(name, batch, h, w, c, k, stride, u8):
    return dict(name=name, kind="depthwise", batch=batch, h=h, w=w, c=c, k=k, stride=stride, u8=u8)


def _fc(name, m, k, o, u8):
    return dict(name=name, kind="fc", m=m, k=k, o=o, u8=u8)


def listed():
    return [
        # interactive classification: one image, nothing to batch it with; latency is all that counts
        _network("mobilenet_v1_b1", "mobilenet_v1", 1),
        # the repository's headline workload: a serving batch that is already resident
        _network("mobilenet_v1_b64", "mobilenet_v1", 64),
        # offline classification of a large collection: the largest batch, throughput only
        _network("mobilenet_v1_b256", "mobilenet_v1", 256),
        # an older uint8 model (per-tensor weights with a zero point), slimmed and at a reduced resolution as such models are
        # deployed, for whatever number of requests was waiting
        _network("mobilenet_v1_w0.75_r160_b13", "mobilenet_v1", 13, resolution=160, width=0.75, weights="per_tensor_u8"),
        # a small serving batch that arrives in and is answered from host memory
        _network("mobilenet_v1_b8_host", "mobilenet_v1", 8, io="host"),
        # the deeper classifier, one image
        _network("resnet50_b1", "resnet50", 1),
        # the deeper classifier at the batch of the repository's second benchmark
        _network("resnet50_b32", "resnet50", 32),
        # the 3x3 layer that dominates the first stage of residual networks
        _conv("conv3x3_56x56x64_b64", 64, 56, 56, 64, 64, 3, 1, False),
        # a down-sampling layer of a mobile detection backbone: channel counts and an extent that are no powers of two
        _conv("conv3x3_s2_75x75x72_120_b9", 9, 75, 75, 72, 120, 3, 2, True),
        # the widest depthwise layer of mobile networks, bound by memory
        _depthwise("depthwise3x3_112x112x32_b64", 64, 112, 112, 32, 3, 1, True),
        # a large classifier or recommender layer for one request: its weights are streamed once
        _fc("fc_4096x4096_m1", 1, 4096, 4096, False),
        # the same layer for a large batch of rows: a matrix product
        _fc("fc_4096x4096_m8192", 8192, 4096, 4096, False),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """Channel counts as networks have them: mostly multiples of 16, the others multiples of 8."""
    step = 16 if rng.random() < 0.7 else 8
    return max(lo, _log(rng, lo, hi) // step * step)


def draw(rng):
    """One more case.  Work stays below that of the largest listed network."""
    pick = rng.random()
    if pick < 0.3:
        return _unnamed(_network("", "mobilenet_v1", _log(rng, 1, 256), resolution=rng.choice([128, 160, 192, 224, rng.randint(97, 224)]),
                                 width=rng.choice([0.5, 0.75, 1.0, 1.0]), weights=rng.choice(["per_channel_s8", "per_channel_s8", "per_tensor_u8"]),
                                 io=rng.choice(["device", "device", "device", "host"])))
    if pick < 0.5:
        return _unnamed(_network("", "resnet50", _log(rng, 1, 32), resolution=rng.choice([160, 192, 224, rng.randint(97, 224)]),
                                 io=rng.choice(["device", "device", "device", "host"])))
    if pick < 0.7:
        while True:
            k = rng.choice([1, 1, 3, 3, 3, 5])
            # output channels now and then are what a head needs (classes, boxes), an odd number
            c = _conv("", _log(rng, 1, 64), 0, 0, _channels(rng, 16, 512), _channels(rng, 16, 512) if rng.random() < 0.8 else rng.randint(17, 300),
                      k, rng.choice([1, 1, 2]), rng.random() < 0.5)
            c["h"] = _log(rng, 7, 112)
            c["w"] = c["h"] if rng.random() < 0.7 else _log(rng, 7, 112)
            if 1e8 <= work(c)["flops"] <= 3e10:
                return _unnamed(c)
    if pick < 0.8:
        while True:
            c = _depthwise("", _log(rng, 1, 64), 0, 0, _channels(rng, 16, 1024), rng.choice([3, 3, 3, 5]), rng.choice([1, 1, 2]), rng.random() < 0.5)
            c["h"] = _log(rng, 7, 112)
            c["w"] = c["h"] if rng.random() < 0.7 else _log(rng, 7, 112)
            if 1e6 <= work(c)["bytes"] <= 1.5e8:
                return _unnamed(c)
    while True:
        c = _fc("", _log(rng, 1, 8192), _log(rng, 256, 4096) // 16 * 16, rng.choice([_log(rng, 10, 4096), _log(rng, 256, 4096) // 64 * 64]), rng.random() < 0.5)
        if work(c)["bytes"] >= 2.5e5:
            return _unnamed(c)


def _unnamed(case):
    case.pop("name")
    return case


# ---- what a program has in hand before the call -----------------------------------------------------------------------
@functools.lru_cache(maxsize=6)
def _definition(net, resolution, width, weights):
    """A model's constants: they belong to the model, not to the images."""
    if net == "resnet50":
        return nets.resnet50(resolution=resolution)
    return nets.mobilenet_v1(resolution=resolution, width=width, weights=weights)


class _Network:
    """A loaded network; its device memory lives as long as somebody holds it or a tensor on it."""

    def __init__(self, net, batch):
        depthwise = any(l.op == "depthwise" for l in net.layers)
        self.dn = DeviceNetwork(net, batch, fuse="auto", lanes=2 if batch >= 16 and batch % 2 == 0 and not depthwise else 1)
        self.net, self.batch = net, batch

    def tensor(self, name):
        """The named activation of the network as a torch tensor on the network's own memory."""
        info = self.net.info(name, self.batch)
        return torch.as_tensor(_OnDevice(self, self.dn.buffers[name].ptr, info), device="cuda")

    def __del__(self):
        self.dn.close()


class _OnDevice:
    def __init__(self, owner, ptr, info):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": info.shape, "typestr": "|u1" if info.dtype == DataType.QAsymmU8 else "|i1", "data": (ptr, False), "version": 2}


def _codes(seed, shape, u8):
    """Activation codes spread over the whole type, on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0 if u8 else -128, 256 if u8 else 128, shape, generator=g, device="cuda", dtype=torch.int16).to(torch.uint8 if u8 else torch.int8)


def _same(size, k, stride):
    out, before, _ = nets.same_padding(size, k, stride)
    return out, before


def _constants(seed, shape, channels, taps, axis, in_scale):
    """Per-channel int8 weights and the int32 bias that goes with them."""
    rng = np.random.default_rng(seed)
    ws = (synth.scales(seed, channels) / np.float32(np.sqrt(taps) / 3.0)).astype(np.float32)
    w = np.clip(np.rint(rng.standard_normal(shape, dtype=np.float32) * 30.0), -127, 127).astype(np.int8)
    return (QTensor(TensorInfo(shape, DataType.QSymmS8, tuple(ws), 0, axis), w),
            QTensor(TensorInfo((channels,), DataType.Signed32, tuple(np.float32(in_scale) * ws), 0, 0), synth.int32_bias(seed, channels)))


def prepare(case, seed):
    if case["kind"] == "network":
        net = _definition(case["net"], case["resolution"], case["width"], case["weights"])
        loaded = _Network(net, case["batch"])
        info = net.info(net.input, case["batch"])
        u8 = info.dtype == DataType.QAsymmU8
        if case["io"] == "host":
            rng = np.random.default_rng(seed)
            images = rng.integers(0 if u8 else -128, 256 if u8 else 128, info.shape, dtype=np.uint8 if u8 else np.int8)
            return {"kind": "host network", "loaded": loaded, "images": QTensor(info, images)}
        loaded.tensor(net.input).copy_(_codes(seed, info.shape, u8))
        return {"kind": "network", "loaded": loaded, "outputs": {"logits": loaded.tensor("logits:out"), "probabilities": loaded.tensor(net.output)}}

    shim.Device()
    u8 = case["u8"]
    dtype, zero = (DataType.QAsymmU8, 128) if u8 else (DataType.QAsymmS8, -3)
    relu6 = dict(activation=shim.ACT_BOUNDED_RELU, act_a=6.0, act_b=0.0)
    if case["kind"] == "fc":
        m, k, o = case["m"], case["k"], case["o"]
        xin, yout = TensorInfo((m, k), dtype, (0.0235,), zero), TensorInfo((m, o), dtype, (0.1,), zero)
        w, b = _constants(seed, (o, k), o, k, 0, 0.0235)
        plan, batch = shim.FullyConnectedPlan(xin, w, b, yout), m
    else:
        dw = case["kind"] == "depthwise"
        ci, co = (case["c"], case["c"]) if dw else (case["ci"], case["co"])
        k, stride = case["k"], case["stride"]
        (ho, pt), (wo, pl) = _same(case["h"], k, stride), _same(case["w"], k, stride)
        batch = case["batch"]
        xin = TensorInfo((batch, case["h"], case["w"], ci), dtype, (0.0235,), zero)
        yout = TensorInfo((batch, ho, wo, co), dtype, (0.0235,), 0 if u8 else -128)
        shape = (1, k, k, co) if dw else (co, k, k, ci)
        w, b = _constants(seed, shape, co, k * k * (1 if dw else ci), 3 if dw else 0, 0.0235)
        plan = shim.Conv2dPlan(xin, w, b, yout, pad_top=pt, pad_left=pl, stride_x=stride, stride_y=stride, depthwise=dw, **relu6)
    x = _codes(seed, xin.shape, u8)
    y = torch.empty(yout.shape, dtype=x.dtype, device="cuda")
    return {"kind": "layer", "plan": plan, "batch": batch, "x": x, "y": y}


def run(state):
    if state["kind"] == "network":
        state["loaded"].dn.enqueue()
        return state["outputs"]
    if state["kind"] == "host network":
        return state["loaded"].dn.run(state["images"]).data
    state["plan"].run(state["batch"], state["x"].data_ptr(), state["y"].data_ptr(), torch.cuda.current_stream().cuda_stream)
    return state["y"]


# ---- what one pass cannot do without ----------------------------------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _network_work(net, resolution, width):
    """(operations per image, bytes in and out per image, bytes of constants) of a network, from its layers' extents."""
    macs, constants, per_image = 0, 0, resolution * resolution * 3

    def conv(size, ci, co, k, stride, depthwise=False):
        nonlocal macs, constants
        out = -(-size // stride)
        taps = k * k * (1 if depthwise else ci)
        macs += out * out * co * taps
        constants += co * taps + 8 * co
        return out

    if net == "resnet50":
        size = conv(resolution, 3, 64, 7, 2)
        size = (size + 1 - 3) // 2 + 1
        ci = 64
        for stage, (c, blocks) in enumerate(zip((64, 128, 256, 512), (3, 4, 6, 3))):
            for i in range(blocks):
                stride = 2 if i == 0 and stage > 0 else 1
                conv(size, ci, c, 1, 1)
                after = conv(size, c, c, 3, stride)
                conv(after, c, 4 * c, 1, 1)
                if i == 0:
                    conv(size, ci, 4 * c, 1, stride)
                size, ci = after, 4 * c
    else:
        wide = lambda c: max(8, int(c * width))
        size, ci = conv(resolution, 3, wide(32), 3, 2), wide(32)
        for co, stride in [(64, 1), (128, 2), (128, 1), (256, 2), (256, 1), (512, 2)] + [(512, 1)] * 5 + [(1024, 2), (1024, 1)]:
            size = conv(size, ci, ci, 3, stride, depthwise=True)
            size = conv(size, ci, wide(co), 1, 1)
            ci = wide(co)
    conv(1, ci, 1001, 1, 1)
    return 2 * macs, per_image + 2 * 1001, constants


def work(case):
    if case["kind"] == "network":
        ops, per_image, constants = _network_work(case["net"], case["resolution"], case["width"])
        return {"bytes": case["batch"] * per_image + constants, "flops": case["batch"] * ops}
    if case["kind"] == "fc":
        m, k, o = case["m"], case["k"], case["o"]
        return {"bytes": m * k + m * o + k * o + 8 * o, "flops": 2 * m * k * o}
    dw = case["kind"] == "depthwise"
    ci, co = (case["c"], case["c"]) if dw else (case["ci"], case["co"])
    k, stride, n = case["k"], case["stride"], case["batch"]
    ho, wo = -(-case["h"] // stride), -(-case["w"] // stride)
    taps = k * k * (1 if dw else ci)
    return {"bytes": n * (case["h"] * case["w"] * ci + ho * wo * co) + co * taps + 8 * co, "flops": 2 * n * ho * wo * co * taps}


def tolerance(case):
    return "exact"
