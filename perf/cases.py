"""The timed work of this framework: what its users run, through the public
entry points (ConvOp, IrBlockSpec, DwPwSpec, SwModel), over the range of sizes,
storage types and options they run it with.

A case is a dict of plain values whose "kind" names the path:
  conv   one convolution through ConvOp: pointwise, K x K or depthwise, with
         an optional residual
  block  one fused inverted-residual block through IrBlockSpec
  dwpw   one fused depthwise 3x3 + pointwise pair through DwPwSpec
  model  a whole .sw model through SwModel: the MobileNetV4-small-width
         segmentation encoder, or the converter's real segmentation model

Activations are NHWC with the channels padded to a multiple of 4 (zeros), as
every entry point takes them; outputs come back in the same layout.
"""
from __future__ import annotations

import json
import struct

import numpy as np
import torch

from ai_engine_amd import conv, sw
from ai_engine_amd import workloads as W

DEV = "cuda:0"
SEGM_FILE = "tests/golden/segm_r11_160x288.sw"  # the reference converter's output for the real model

DT = {"f32": conv.DType.F32, "f16": conv.DType.F16, "bf16": conv.DType.BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
NBYTES = {"f32": 4, "f16": 2, "bf16": 2}
ACT = {a.name.lower(): a for a in conv.Activation}


def c4(c):
    return -(-c // 4) * 4


# ---------------------------------------------------------------- the cases

def _conv(name, n, h, w, cin, cout, k=1, s=1, dw=False, act="relu", res=False, dt="f32"):
    c = dict(name=name) if name else {}
    return c | dict(kind="conv", n=n, h=h, w=w, cin=cin, cout=cout, k=k, s=s, dw=dw, act=act, res=res, dt=dt)


def listed():
    return [
        # one frame's deepest pointwise layer (a skinny GEMM, 180 pixels): a
        # single-frame user's smallest call, where latency is all there is
        _conv("pw_960to160_10x18_b1_f32", 1, 10, 18, 960, 160, act="none"),
        # the same layer for an offline job's batch: the largest fp32 GEMM
        _conv("pw_960to160_10x18_b256_f32", 256, 10, 18, 960, 160, act="none"),
        # an expand of a wide model run op by op in 16 bit, at an odd frame size
        _conv("pw_192to768_21x37_b64_f16", 64, 21, 37, 192, 768, act="hardswish", dt="f16"),
        # a downsampling 3x3 near the input: few channels, many pixels
        _conv("conv3x3s2_16to32_160x288_b32_f32", 32, 160, 288, 16, 32, k=3, s=2),
        # a decoder's or backbone's dense 3x3 with residual in 16 bit
        _conv("conv3x3_128to128_40x72_b32_f16", 32, 40, 72, 128, 128, k=3, res=True, dt="f16"),
        # a depthwise layer on its own, as an unfused graph runs it
        _conv("dw3x3s2_128_80x144_b32_f16", 32, 80, 144, 128, 128, k=3, s=2, dw=True, dt="f16"),
        # a MobileNet block at mid resolution for a serving batch
        dict(name="block_64_256_64_40x72_b64_f16", kind="block", n=64, h=40, w=72, cin=64, cexp=256, cout=64, s=1,
             res=True, dt="f16"),
        # a late block for a few frames: small launches, wide layers
        dict(name="block_128_512_128_10x18_b8_bf16", kind="block", n=8, h=10, w=18, cin=128, cexp=512, cout=128, s=1,
             res=True, dt="bf16"),
        # the second half of an fp32 block (fp32 blocks run as expand + this)
        dict(name="dwpw_256to64_40x72_b64_f32", kind="dwpw", n=64, h=40, w=72, c=256, cout=64, s=1, res=True,
             dt="f32"),
        # offline throughput: the whole encoder on a resident batch, tuned at load
        dict(name="encoder_160x288_b64_f16", kind="model", model="encoder", n=64, dt="f16", tune=True, host=False),
        # one camera frame through the real model, host memory in and out
        dict(name="segm_160x288_b1_f32_host", kind="model", model="segm", n=1, dt="f32", tune=False, host=True),
        # the same model for a serving batch on the device, 16-bit storage
        dict(name="segm_160x288_b64_f16", kind="model", model="segm", n=64, dt="f16", tune=False, host=False),
    ]


def _logint(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _frame(rng, lo, hi):
    """A frame size: one of the models' own, or any (odd ones too)."""
    own = [(160, 288), (80, 144), (40, 72), (20, 36), (10, 18)]
    if rng.random() < 0.5:
        fits = [f for f in own if lo <= f[0] <= hi]
        return rng.choice(fits)
    h = _logint(rng, lo, hi)
    return h, max(8, int(h * rng.uniform(1.0, 1.8)))


# a drawn case's bound: the work of the largest listed cases (flops by
# storage type, bytes)
_MAX_FLOPS = {"f32": 1.4e10, "f16": 9.0e10, "bf16": 9.0e10}
_MAX_BYTES = 4.0e8


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        dense = _MAX_FLOPS[c["dt"]] if c["kind"] in ("block", "model") else min(_MAX_FLOPS[c["dt"]], 4e10)
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= dense:
            return c


def _draw(rng):
    kind = rng.choice(["pw", "pw", "conv", "conv", "dw", "block", "block", "dwpw", "model"])
    if kind == "model":
        model = rng.choice(["encoder", "segm"])
        host = rng.random() < 0.3
        dt = rng.choice(["f16", "f16", "bf16", "f32"] if model == "segm" else ["f16", "f16", "bf16"])
        n = _logint(rng, 1, 4) if host else _logint(rng, 1, 64)
        return dict(kind="model", model=model, n=n, dt=dt, tune=model == "encoder", host=host)
    dt = rng.choice(["f32", "f16", "f16", "bf16"])
    n = _logint(rng, 1, 64)
    if kind == "pw":
        h, w = _frame(rng, 8, 80)
        cin, cout = (rng.choice([16, 24, 32, 44, 48, 64, 72, 96, 128, 192, 240, 320, 576, 960]) for _ in range(2))
        act = rng.choice(["none", "relu", "relu6", "hardswish"])
        return _conv(None, n, h, w, cin, cout, act=act, res=rng.random() < 0.3, dt=dt)
    if kind == "conv":
        h, w = _frame(rng, 10, 160)
        s = rng.choice([1, 1, 2])
        cin, cout = (rng.choice([16, 24, 32, 48, 64, 72, 96, 128, 160, 256]) for _ in range(2))
        k = rng.choice([3, 3, 3, 5])
        act = rng.choice(["none", "relu", "hardswish"])
        return _conv(None, n, h, w, cin, cout, k=k, s=s, act=act, res=rng.random() < 0.3, dt=dt)
    if kind == "dw":
        h, w = _frame(rng, 10, 160)
        c = rng.choice([32, 44, 64, 96, 128, 256, 384])
        return _conv(None, n, h, w, c, c, k=rng.choice([3, 3, 5]), s=rng.choice([1, 2]), dw=True, dt=dt)
    if kind == "block":
        h, w = _frame(rng, 10, 80)
        cin, cout, s = rng.choice([(32, 32, 1), (32, 64, 2), (48, 48, 1), (64, 64, 1), (64, 96, 2), (96, 96, 1),
                                   (96, 128, 2), (128, 128, 1)])
        cexp = cin * (2 if cin == 48 else 4)
        return dict(kind="block", n=n, h=h, w=w, cin=cin, cexp=cexp, cout=cout, s=s, res=cin == cout,
                    dt=rng.choice(["f16", "bf16"]))
    h, w = _frame(rng, 10, 80)
    c = rng.choice([44, 48, 96, 128, 192, 256])
    return dict(kind="dwpw", n=n, h=h, w=w, c=c, cout=rng.choice([24, 32, 48, 64]), s=rng.choice([1, 1, 2]),
                res=rng.random() < 0.3, dt=rng.choice(["f32", "f16"]))


# ---------------------------------------------------------------- descriptors

def _conv_op(c):
    p = c["k"] // 2
    return conv.ConvOp(ih=c["h"], iw=c["w"], cin=c["cin"], cout=c["cout"], kh=c["k"], kw=c["k"], sh=c["s"], sw=c["s"],
                       pad=(p,) * 4, groups=c["cin"] if c["dw"] else 1, act=ACT[c["act"]], residual=c["res"],
                       dt=DT[c["dt"]], n=c["n"])


def _block_spec(c):
    return conv.IrBlockSpec(ih=c["h"], iw=c["w"], cin=c["cin"], cexp=c["cexp"], cout=c["cout"], s=c["s"],
                            residual=c["res"], dt=DT[c["dt"]], n=c["n"])


def _dwpw_spec(c):
    return conv.DwPwSpec(ih=c["h"], iw=c["w"], c=c["c"], cout=c["cout"], s=c["s"], residual=c["res"],
                         dt=DT[c["dt"]], n=c["n"])


def _model_bytes(c, seed):
    if c["model"] == "segm":
        with open(SEGM_FILE, "rb") as f:
            return f.read()
    layers, meta = W.mnv4_small_encoder_160x288(c["n"])
    return sw.conv_graph_to_sw("encoder", layers, W.make_weights(layers, seed=seed), meta["h"], meta["w"], meta["c"])


# ---------------------------------------------------------------- inputs

class _Draws:
    """Seeded values: activations on the device, weights on the host."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.r = np.random.default_rng(seed)

    def act(self, n, h, w, c, dt, relu):
        """Activations as a layer meets them: after a ReLU (half of them
        zero) or linear; padding channels zero."""
        x = torch.randn(n, h, w, c4(c), generator=self.g, device=DEV)
        if relu:
            x.clamp_(min=0)
        x[..., c:] = 0
        return x.to(TORCH[dt])

    def weight(self, cout, cin, k):
        """He-initialised OIHW weights (cin 1 for a depthwise)."""
        return (self.r.standard_normal((cout, cin, k, k)) * np.sqrt(2.0 / (k * k * cin))).astype(np.float32)

    def bias(self, c):
        return (self.r.standard_normal(c) * 0.1).astype(np.float32)


def _inputs(c, seed):
    """x, residual (or None) and [(weights, bias, depthwise)] of a conv, block or dwpw case."""
    d = _Draws(seed)
    n, h, w, dt = c["n"], c["h"], c["w"], c["dt"]
    if c["kind"] == "conv":
        oh, ow = _conv_op(c).out_hw()
        x = d.act(n, h, w, c["cin"], dt, relu=True)
        res = d.act(n, oh, ow, c["cout"], dt, relu=False) if c["res"] else None
        return x, res, [(d.weight(c["cout"], 1 if c["dw"] else c["cin"], c["k"]), d.bias(c["cout"]), c["dw"])]
    if c["kind"] == "block":
        x = d.act(n, h, w, c["cin"], dt, relu=False)  # the linear output of the block before it
        e = c["cexp"]
        return x, x if c["res"] else None, [(d.weight(e, c["cin"], 1), d.bias(e), False),
                                            (d.weight(e, 1, 3), d.bias(e), True),
                                            (d.weight(c["cout"], e, 1), d.bias(c["cout"]), False)]
    oh, ow = _dwpw_spec(c).out_hw()
    x = d.act(n, h, w, c["c"], dt, relu=True)
    res = d.act(n, oh, ow, c["cout"], dt, relu=False) if c["res"] else None
    return x, res, [(d.weight(c["c"], 1, 3), d.bias(c["c"]), True),
                    (d.weight(c["cout"], c["c"], 1), d.bias(c["cout"]), False)]


def _upload(a):
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).to(DEV)


def _packed(wb, dt):
    """Device copies of the packed weights and bias of one conv, as a loader makes them."""
    w, b, dw = wb
    cout, cin, k, _ = w.shape
    if dw:
        p = conv.pack_weights_dw(w.ravel(), cout, k, k, DT[dt])
    else:
        p, _ = conv.pack_weights_conv(w.ravel(), cout, cin, k, k, 4, DT[dt])
    return _upload(p), _upload(conv.pack_bias(b, cout, DT[dt]))


class _DeviceArray:
    """A device buffer of `owner`, for torch.as_tensor: the tensor made from
    it keeps this object, and with it the owner of the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _model_output(m):
    """The model's output tensor where it lies on the device (NHWC-C4)."""
    t = m.tensor(m.outputs[0])
    shape = (t.n, t.h, t.w, t.stride_c)
    if t.dt == conv.DType.F32:
        return torch.as_tensor(_DeviceArray(m, t.data, shape, "<f4"), device=DEV)
    y = torch.as_tensor(_DeviceArray(m, t.data, shape, "<i2"), device=DEV)
    return y.view(torch.float16 if t.dt == conv.DType.F16 else torch.bfloat16)


def _frames(c, seed):
    """Camera frames scaled to [-1, 1): a smooth scene with noise on it."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    low = torch.rand(c["n"], 3, 10, 18, generator=g, device=DEV) * 1.6 - 0.8
    x = torch.nn.functional.interpolate(low, size=(160, 288), mode="bilinear", align_corners=False)
    x = x + (torch.rand(x.shape, generator=g, device=DEV) * 0.4 - 0.2)
    return x.permute(0, 2, 3, 1).contiguous()


def prepare(case, seed):
    c = case
    st = {"case": c}
    if c["kind"] == "model":
        m = sw.SwModel(_model_bytes(c, seed), n=c["n"], dt=DT[c["dt"]] if c["dt"] != "f32" else None, tune=c["tune"])
        x = _frames(c, seed)
        st.update(model=m, x=x.cpu().numpy() if c["host"] else x)
        if not c["host"]:
            st["y"] = _model_output(m)
        return st
    x, res, wbs = _inputs(c, seed)
    st.update(x=x, res=res, w=[t for wb in wbs for t in _packed(wb, c["dt"])])
    if c["kind"] == "conv":
        st["op"] = op = _conv_op(c)
        nb = op.workspace_bytes()
        st["ws"] = torch.empty(nb // 4, dtype=torch.float32, device=DEV) if nb else None
        cout = c["cout"]
    else:
        st["op"] = op = _block_spec(c) if c["kind"] == "block" else _dwpw_spec(c)
        cout = c["cout"]
    oh, ow = op.out_hw()
    st["y"] = torch.empty(c["n"], oh, ow, c4(cout), dtype=TORCH[c["dt"]], device=DEV)
    return st


def run(state):
    st = state
    c = st["case"]
    if c["kind"] == "model":
        m = st["model"]
        m.upload_input(m.inputs[0], st["x"])
        m.infer()
        return m.read_output() if c["host"] else st["y"]
    if c["kind"] == "conv":
        return st["op"].run(st["x"], *st["w"], st["res"], st["y"], ws=st["ws"])
    return st["op"].run(st["x"], *st["w"], st["res"], st["y"])


# ---------------------------------------------------------------- work

def _graph(data):
    """The graph and weight blob of a .sw container."""
    _, _, align, joff, jlen = struct.unpack_from("<IIIQQ", data, 4)
    off = -(-(joff + jlen) // max(align, 1)) * max(align, 1)
    return json.loads(data[joff:joff + jlen]), data[off:]


def _model_work(c):
    """A model's conv flops, and the frames in, the result out and the weights once."""
    if c["model"] == "encoder":
        layers, _ = W.mnv4_small_encoder_160x288(c["n"])
        flops = sum(L.flops(c["n"]) for L in layers)
        params = sum(L.k * L.k * (1 if L.depthwise else L.cin) * L.cout + L.cout for L in layers)
        out = layers[-1].out_hw() + (layers[-1].cout,)
    else:
        with open(SEGM_FILE, "rb") as f:
            g, _ = _graph(f.read())
        T, flops, params = g["tensors"], 0, 0
        for o in g["ops"]:
            if o["kind"] == "conv":
                per = o["kh"] * o["kw"] * o["cin"] // o["groups"] * o["cout"]
                flops += 2 * c["n"] * T[o["out"]]["h"] * T[o["out"]]["w"] * per
                params += per + o["cout"]
        t = T[g["outputs"][0]]
        out = (t["h"], t["w"], t["c"])
    b = NBYTES[c["dt"]]
    ob = 4 if c["host"] else b
    return {"bytes": c["n"] * (160 * 288 * 3 * 4 + out[0] * out[1] * out[2] * ob) + params * b, "flops": flops}


def work(case):
    c = case
    if c["kind"] == "model":
        return _model_work(c)
    b, n = NBYTES[c["dt"]], c["n"]
    if c["kind"] == "conv":
        oh, ow = _conv_op(c).out_hw()
        per = c["k"] ** 2 * (1 if c["dw"] else c["cin"])
        cin, cout, wts = c["cin"], c["cout"], per * c["cout"] + c["cout"]
        macs = oh * ow * per * cout
    elif c["kind"] == "block":
        oh, ow = _block_spec(c).out_hw()
        cin, e, cout = c["cin"], c["cexp"], c["cout"]
        wts = cin * e + 9 * e + e * cout + 2 * e + cout
        macs = c["h"] * c["w"] * cin * e + oh * ow * (9 * e + e * cout)
    else:
        oh, ow = _dwpw_spec(c).out_hw()
        cin, cout = c["c"], c["cout"]
        wts = 9 * cin + cin * cout + cin + cout
        macs = oh * ow * (9 * cin + cin * cout)
    out = oh * ow * cout
    res = out if c["res"] and c["kind"] != "block" else 0  # a block's residual is its input
    return {"bytes": b * (n * (c["h"] * c["w"] * cin + out + res) + wts), "flops": 2 * n * macs}


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times the error against exact() measured over the declared
    ranges. fp32: 1e-7 to 4e-7 for single layers (the longest K the most),
    1.3e-6 through the whole model. 16 bit: the rounding of the result
    (2.1e-4 f16, 1.7e-3 bf16), in blocks and pairs of the stored
    intermediates too (3.6e-4 / 2.9e-3), in models of every layer."""
    c = case
    if c["kind"] == "model":
        rel = {"encoder": {"f32": 5e-6, "f16": 7e-3, "bf16": 5e-2}, "segm": {"f32": 5e-6, "f16": 1e-2, "bf16": 9e-2}}
        return {"rel": rel[c["model"]][c["dt"]]}
    if c["dt"] == "f32":
        return {"rel": 2e-6}
    rel = 8e-4 if c["kind"] == "conv" else 1.4e-3
    return {"rel": rel if c["dt"] == "f16" else 8 * rel}


# ---------------------------------------------------------------- exact

def _act64(name, v):
    if name == "none":
        return v
    if name == "relu":
        return v.clamp(min=0)
    if name == "relu6":
        return v.clamp(0, 6)
    if name == "hardswish":
        return v * (v / 6 + 0.5).clamp(0, 1)
    if name == "sigmoid":
        return torch.sigmoid(v)
    raise ValueError(name)


def _conv64(x, w, b, k, s, p, dw):
    """NHWC convolution in 64 bits: x [n,h,w,cin], w [cout,cin or 1,k,k]."""
    n, h, wd, ci = x.shape
    oh, ow = (h + 2 * p - k) // s + 1, (wd + 2 * p - k) // s + 1
    co = w.shape[0]
    w = torch.from_numpy(np.ascontiguousarray(w)).to(DEV).double()
    y = torch.from_numpy(b).to(DEV).double().expand(n, oh, ow, co).clone()
    for ky in range(k):
        for kx in range(k):
            # the outputs whose tap (ky, kx) falls inside the image
            y0, x0 = max(0, -(-(p - ky) // s)), max(0, -(-(p - kx) // s))
            y1, x1 = min(oh, (h - 1 + p - ky) // s + 1), min(ow, (wd - 1 + p - kx) // s + 1)
            if y1 <= y0 or x1 <= x0:
                continue
            iy, ix = y0 * s + ky - p, x0 * s + kx - p
            t = x[:, iy:iy + (y1 - y0 - 1) * s + 1:s, ix:ix + (x1 - x0 - 1) * s + 1:s]
            if dw:
                y[:, y0:y1, x0:x1] += t * w[:, 0, ky, kx]
            else:
                m = t.reshape(-1, ci) @ w[:, :, ky, kx].t().contiguous()
                y[:, y0:y1, x0:x1] += m.view(n, y1 - y0, x1 - x0, co)
    return y


def _stored(a, dt):
    """Host values as the storage type holds them."""
    return a if dt == "f32" else torch.from_numpy(a).to(TORCH[dt]).float().numpy()


def _pad_channels(y):
    return torch.nn.functional.pad(y, (0, c4(y.shape[-1]) - y.shape[-1]))


def _blob_f32(blob, ref):
    return np.frombuffer(blob, np.float32, ref["len"] // 4, ref["off"])


def _sw_weights(blob, o, dt):
    """OIHW weights and bias of a graph's conv, unpacked from the converter's layout."""
    co, ci, kh, kw = o["cout"], o["cin"], o["kh"], o["kw"]
    p = _blob_f32(blob, o["w"])
    if o["groups"] > 1:  # [tap][channel group][4]
        w = p.reshape(kh * kw, -1)[:, :co].T.reshape(co, 1, kh, kw)
    else:  # [tap][input group][output group][output][input]
        v = p.reshape(kh * kw, o["kg_pad"], -(-co // 4), 4, 4)
        w = v.transpose(2, 3, 1, 4, 0).reshape(c4(co), -1, kh * kw)[:co, :ci].reshape(co, ci, kh, kw)
    return _stored(np.ascontiguousarray(w), dt), _stored(_blob_f32(blob, o["b"])[:co].copy(), dt)


def _resize64(x, oh, ow):
    """Half-pixel bilinear resize of NHWC values."""
    def taps(o, size):
        f = (torch.arange(o, device=DEV, dtype=torch.float64) + 0.5) * size / o - 0.5
        i = f.floor()
        return i.long().clamp(0, size - 1), (i.long() + 1).clamp(0, size - 1), f - i

    y0, y1, ty = taps(oh, x.shape[1])
    x0, x1, tx = taps(ow, x.shape[2])
    ty, tx = ty.view(1, -1, 1, 1), tx.view(1, 1, -1, 1)
    top = x[:, y0][:, :, x0] * (1 - tx) + x[:, y0][:, :, x1] * tx
    bot = x[:, y1][:, :, x0] * (1 - tx) + x[:, y1][:, :, x1] * tx
    return top * (1 - ty) + bot * ty


def _sw64(data, x, dt):
    """A .sw graph in 64 bits, its weights as stored in dt."""
    g, blob = _graph(data)
    T = g["tensors"]
    last = {}
    for i, o in enumerate(g["ops"]):
        for v in [o.get("in"), o.get("res"), o.get("a"), *(p["in"] for p in o.get("srcs", []) + o.get("parts", [])),
                  *(v.get("tid") for v in o.get("b", {}).values() if isinstance(v, dict))]:
            last[v] = i
    out = g["outputs"][0]
    base = T[out]["alias"]["of"] if T[out]["alias"] else out
    vals = {g["inputs"][0]: x}
    for i, o in enumerate(g["ops"]):
        if o["kind"] == "conv":
            src = torch.cat([vals[p["in"]] for p in o["srcs"]], -1) if o.get("srcs") else vals[o["in"]]
            y = _conv64(src, *_sw_weights(blob, o, dt), o["kh"], o["sh"], o["pad"][0], o["groups"] > 1)
            y = _act64(o["act"], y)
            if o["res"] is not None:
                y = y + vals[o["res"]]
        elif o["kind"] == "gpool":
            y = vals[o["in"]].mean((1, 2), keepdim=True)
        elif o["kind"] == "binary":
            (b,) = o["b"].values()
            y = vals[o["a"]] * vals[b["tid"]] if o["op"] == "mul" else vals[o["a"]] + vals[b["tid"]]
        elif o["kind"] == "resize":
            y = _resize64(vals[o["in"]], o["oh"], o["ow"])
        else:  # concat
            y = torch.cat([vals[p["in"]] for p in o["parts"]], -1)
        vals[o["out"]] = y
        for t in [t for t in vals if last.get(t, -1) <= i and t != base and t != o["out"]]:
            del vals[t]
    return vals[base]


def exact(case, seed):
    c = case
    if c["kind"] == "model":
        y = _sw64(_model_bytes(c, seed), _frames(c, seed).double(), c["dt"])
        return y.cpu().numpy() if c["host"] else _pad_channels(y)
    x, res, wbs = _inputs(c, seed)
    wbs = [(_stored(w, c["dt"]), _stored(b, c["dt"]), dw) for w, b, dw in wbs]
    cin = c["c"] if c["kind"] == "dwpw" else c["cin"]
    y = x[..., :cin].double()
    r = None if res is None else res[..., :c["cout"]].double()
    if c["kind"] == "conv":
        (w, b, dw), = wbs
        y = _act64(c["act"], _conv64(y, w, b, c["k"], c["s"], c["k"] // 2, dw))
    else:
        acts = ["relu", "relu", "none"] if c["kind"] == "block" else ["relu", "none"]
        for (w, b, dw), act in zip(wbs, acts):
            y = _act64(act, _conv64(y, w, b, 3 if dw else 1, c["s"] if dw else 1, 1 if dw else 0, dw))
    if r is not None:
        y = y + r
    return _pad_channels(y)
