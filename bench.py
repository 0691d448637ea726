"""Benchmark of the MI355X conv-as-GEMM backend (one GPU).

Headline workload (value, frames/s): the MobileNetV4-small-width segmentation
encoder at 160x288, batch 64, f16 storage with fp32 accumulation -- 32 convs
(stem 3x3 s2 3->32, ten inverted-residual blocks, 1x1 head 128->2) with
random He-init weights and U[-1,1) synthetic input already resident in HBM.
One step = all 32 convs from the resident logical NHWC fp32 input: the stem
reads it directly and rounds each value to the storage dtype as it loads it
(no separate pack launch).

Also measured in the same run (the "kernels" object), each with absolute
TFLOP/s, GB/s and its roofline fraction (t_roof / t_measured,
t_roof = max(flops / MFMA peak, bytes / 8 TB/s)):
  pw_32to64_relu6_80x144            1x1 32->64 + ReLU6, [1,80,144,32] fp32
  pw_960to160_10x18_b1_splitk{1,4,8} 1x1 960->160, [1,10,18,960] fp32, split-K forced
  pw_960to160_10x18_b256[_splitk{1,4,8}] the same layer at batch 256 (policy: the
                                     LDS-streamed GEMM, no split; forced 1/4/8)
  igemm3x3s2_16to32_relu_160x288_b32 3x3 s2 pad 1 16->32 + ReLU, [32,160,288,16] fp32
  igemm3x3s1_32to64_relu_80x144_b32  3x3 s1 pad 1 32->64 + ReLU, [32,80,144,32] fp32
  ir_block_chain_4x_64c_40x72_b64    4 inverted-residual blocks at [64,40,72,64] fp32
  encoder_bf16                       the headline workload with bf16 storage
Small configurations are timed over rotated buffer sets larger than the 256 MB
Infinity Cache, so their GB/s are HBM figures.

cpu_baseline: the oracle's C restatement of ai-cpu (the reference's CPU path:
conv_std / im2row stem / conv_dw / pw_dot head, row-band threads) running the
same encoder in fp32 on the host's cores, on a bounded sample of frames.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--dtype bf16|f16]
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

METRIC = "conv-GEMM TFLOP/s + HBM GB/s (% roofline), frames/s at 160x288 batch 64"
HBM_GBS = 8000.0
PEAK_TF = {"f32": 157.3, "f16": 2516.6, "bf16": 2516.6}
MALL_BYTES = 256 << 20


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def roof(flops: float, nbytes: float, secs: float, dtype: str) -> dict:
    t_mfma = flops / (PEAK_TF[dtype] * 1e12)
    t_hbm = nbytes / (HBM_GBS * 1e9)
    bound = "mfma" if t_mfma >= t_hbm else "hbm"
    return dict(
        us=secs * 1e6, tflops=flops / secs / 1e12, gbs=nbytes / secs / 1e9, bound=bound,
        frac=max(t_mfma, t_hbm) / secs, flops=flops, bytes=nbytes,
    )


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--dtype", default="f16", choices=["bf16", "f16"])
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-kernels", action="store_true", help="skip the per-config kernel table")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--choices", default=None,
                    help="JSON map block -> launch label (as printed in block_choices) to load without tuning")
    ap.add_argument("--profile-config", default=None, choices=sorted(PROFILE_CONFIGS),
                    help="run only this workload's launches, --profile-reps times, and print no JSON line "
                         "(the command rocprofv3 counter passes run)")
    ap.add_argument("--profile-reps", type=int, default=20)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU; --gpus {args.gpus} is not supported "
              "(batch sharding across GPUs needs no exchange and is not run here)", file=sys.stderr)
        return 2

    import numpy as np
    import torch

    from ai_engine_amd import conv, workloads as W
    from ai_engine_amd.model import Model

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda:0")
    conv.lib()
    torch.manual_seed(0)
    DT = {"f32": conv.DType.F32, "f16": conv.DType.F16, "bf16": conv.DType.BF16}
    if args.profile_config:
        return profile_config(args, torch, conv, W, Model, dev, DT)

    # ------------------------------------------------------------ headline: encoder, batch 64
    layers, meta = W.mnv4_small_encoder_160x288(64)
    n, H, Wd = meta["n"], meta["h"], meta["w"]
    wts = W.make_weights(layers, seed=0)
    x = (torch.rand(n, H, Wd, 3, device=dev) * 2 - 1).contiguous()
    model = Model(layers, wts, n, H, Wd, 3, dt=DT[args.dtype],
                  choices=json.loads(args.choices) if args.choices else None)
    stream = torch.cuda.current_stream()
    log("load-time block choices: " + ", ".join(f"{k} {v[0]} ({v[1]:.1f} us)" for k, v in model.choices.items()))

    def step():
        model.upload_input(x)
        model.infer()

    # per-step distribution first (untimed for the headline): max(100, K)
    # steps, each bracketed by HIP events
    NS = max(100, args.steps)
    sev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(NS)]
    for a, b in sev:
        a.record(stream)
        step()
        b.record(stream)
    torch.cuda.synchronize()
    st = sorted(a.elapsed_time(b) for a, b in sev)
    step_stats = {"steps": NS, "min_ms": round(st[0], 4), "median_ms": round(st[NS // 2], 4),
                  "max_ms": round(st[-1], 4), "frames_per_s_at_median": round(n / (st[NS // 2] / 1e3), 1)}
    log(f"per-step (events, {NS} steps): min {st[0]:.3f} median {st[NS // 2]:.3f} max {st[-1]:.3f} ms")
    # the headline: W warm-up steps, then exactly K steps between a
    # synchronize on either side
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    e0.record(stream)
    for _ in range(args.steps):
        step()
    e1.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    gpu_ms = e0.elapsed_time(e1) / args.steps
    ms_per_step = wall * 1e3 / args.steps
    fps = n / (ms_per_step / 1e3)
    log(f"encoder {args.dtype} b{n}: {ms_per_step:.3f} ms/step wall, {gpu_ms:.3f} ms/step gpu, {fps:.0f} frames/s")

    # per-op timing, grouped by kernel instantiation: R passes over the step,
    # HIP events on the launch stream around every launch (each median over
    # the passes). An event pair adds its own few microseconds to a launch;
    # the dominant kernel is timed again below with fewer events.
    R = 5
    nops = len(model.ops)
    evs = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(nops)]
           for _ in range(R)]
    for r in range(R):
        model.upload_input(x)
        for i in range(nops):
            evs[r][i][0].record(stream)
            model.launch_op(i)
            evs[r][i][1].record(stream)
    torch.cuda.synchronize()
    op_secs = [sorted(evs[r][i][0].elapsed_time(evs[r][i][1]) for r in range(R))[R // 2] / 1e3 for i in range(nops)]
    act_b = 2 if args.dtype != "f32" else 4
    groups: dict[str, dict] = {}
    layer_rows = []
    for i, op in enumerate(model.ops):
        t = op_secs[i]
        fl, by = op.flops(n), op.bytes(n, act_b, act_b)
        key = kernel_key(conv, op, n, DT[args.dtype], args.dtype)
        g = groups.setdefault(key, dict(launches=0, secs=0.0, flops=0, bytes=0, grids=[]))
        g["launches"] += 1
        if op.kind in ("ir_block", "stem_ir_block", "ir_block_head"):
            pl = op.spec.plan()
            # dispatch size in threads, as rocprofv3 lists it
            g["grids"].append(pl.grid * 64 * pl.waves)
        g["secs"] += t
        g["flops"] += fl
        g["bytes"] += by
        layer_rows.append(dict(op=op.name, kernel=key, us=round(t * 1e6, 2),
                               gbs=round(by / t / 1e9, 1), tflops=round(fl / t / 1e12, 2)))
    # the step's own roofline: every launch at its binding roof with the bytes
    # it must move (a fused block's expanded tensors never reach HBM)
    fused_roof_s = sum(max(op.flops(n) / (PEAK_TF[args.dtype] * 1e12), op.bytes(n, act_b, act_b) / (HBM_GBS * 1e9))
                       for op in model.ops)
    fused_bytes = sum(op.bytes(n, act_b, act_b) for op in model.ops)
    dom_key, dom = max(groups.items(), key=lambda kv: kv[1]["secs"])
    # the dominant kernel in the step: its launches are consecutive ops (the
    # encoder's b0, b1), so whole steps run with one event pair around that
    # run of launches only -- one event overhead per run rather than per
    # launch, every other launch of the step as in the timed steps
    dom_ops = [i for i, op in enumerate(model.ops) if kernel_key(conv, op, n, DT[args.dtype], args.dtype) == dom_key]
    dom_timing = "HIP events around each launch, median of 5 passes over the step"
    if dom_ops == list(range(dom_ops[0], dom_ops[-1] + 1)):
        RS = 20
        ev2 = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(RS)]
        for r in range(RS):
            model.upload_input(x)
            for i in range(nops):
                if i == dom_ops[0]:
                    ev2[r][0].record(stream)
                model.launch_op(i)
                if i == dom_ops[-1]:
                    ev2[r][1].record(stream)
        torch.cuda.synchronize()
        run = sorted(a.elapsed_time(b) for a, b in ev2)[RS // 2] / 1e3
        dom["secs"] = run
        dom_timing = (f"in the step: one HIP event pair around its {len(dom_ops)} consecutive launches (ops "
                      f"{dom_ops[0]}..{dom_ops[-1]}), every other launch of the step as timed, median of {RS} "
                      "steps, divided by the launches")
    dr = roof(dom["flops"] / dom["launches"], dom["bytes"] / dom["launches"], dom["secs"] / dom["launches"],
              args.dtype)
    if dr["bound"] == "hbm":
        roofline = dict(bound="hbm", achieved=round(dr["gbs"], 1), peak=HBM_GBS, unit="GB/s",
                        frac=round(dr["gbs"] / HBM_GBS, 4), traffic=None)
    else:
        roofline = dict(bound="mfma", achieved=round(dr["tflops"], 2), peak=PEAK_TF[args.dtype], unit="TFLOP/s",
                        frac=round(dr["tflops"] / PEAK_TF[args.dtype], 4), traffic=None)
    roofline["traffic"] = measured_traffic(dom_key)
    roofline.update(kernel=dom_key, launches_per_step=dom["launches"], dispatch_threads=sorted(dom["grids"]),
                    avg_launch_us=round(dom["secs"] / dom["launches"] * 1e6, 2),
                    timing=dom_timing,
                    algorithmic_bytes_per_launch=int(dom["bytes"] / dom["launches"]),
                    algorithmic_flops_per_launch=int(dom["flops"] / dom["launches"]),
                    share_of_step=round(dom["secs"] / (gpu_ms / 1e3), 3))
    tot_fl, tot_by = W.totals(layers, n, act_b, act_b)
    unfused_roof_s = sum(max(L.flops(n) / (PEAK_TF[args.dtype] * 1e12), L.bytes(n, act_b, act_b) / (HBM_GBS * 1e9))
                         for L in layers)
    log(f"dominant kernel {dom_key}: {roofline}")

    # plain device copy of 1 GiB (the calibration kernel for HBM counters and
    # the bandwidth a streaming kernel can reach on this box)
    src_buf = torch.empty(1 << 28, dtype=torch.float32, device=dev)
    dst_buf = torch.empty_like(src_buf)
    t_copy = time_launches(torch, stream, lambda r: dst_buf.copy_(src_buf), 10)
    copy_gbs = 2 * src_buf.numel() * 4 / t_copy / 1e9
    del src_buf, dst_buf
    log(f"device copy 1 GiB: {copy_gbs:.0f} GB/s")

    # ------------------------------------------------------------ per-config kernel table (fp32)
    kernels = {}
    if not args.no_kernels:
        kernels = kernel_table(torch, conv, W, Model, dev, stream, DT)
        kernels.update(real_model(torch, conv, dev, stream))
        kernels["encoder_f16" if args.dtype == "bf16" else "encoder_bf16"] = encoder_other(
            torch, W, Model, layers, wts, x, n, H, Wd, "f16" if args.dtype == "bf16" else "bf16", DT, stream)
    kernels["encoder_layers"] = layer_rows
    kernels["encoder_via_aih_model"] = encoder_native(torch, W, layers, wts, x, n, H, Wd, DT[args.dtype], stream,
                                                      fps)
    kernels["encoder_block_choices"] = {k: {"choice": v[0], "us": round(v[1], 2)} for k, v in model.choices.items()}

    # ------------------------------------------------------------ CPU baseline (oracle ai-cpu restatement)
    cpu = None
    if not args.no_cpu:
        model.upload_input(x)
        model.infer()
        torch.cuda.synchronize()
        y0 = model.read_output().reshape(n, -1)[0]
        x0 = x[0].contiguous().cpu().numpy().ravel()
        cpu = cpu_baseline(layers, wts, H, Wd, args.cpu_seconds, W=W, parity_in=(x0, y0, args.dtype))

    out = {
        "metric": METRIC, "value": round(fps, 1), "unit": "frames/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_per_step, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": args.dtype, "data": "synthetic",
        "config": {"workload": meta["name"], "batch": n, "height": H, "width": Wd, "convs": len(layers),
                   "storage": args.dtype, "accumulate": "f32", "step": "32 convs from the resident fp32 NHWC input (the stem rounds it to the storage dtype as it reads)"},
        "gpu_ms_per_step": round(gpu_ms, 4),
        "step_stats": step_stats,
        "step_roofline_fused": {"roof_us": round(fused_roof_s * 1e6, 1), "bytes": fused_bytes,
                                "flops": sum(op.flops(n) for op in model.ops),
                                "frac": round(fused_roof_s / (gpu_ms / 1e3), 4),
                                "note": "the step's own roofline: sum over the launches it runs of max(flops / "
                                        "MFMA peak, bytes / 8 TB/s), each launch counting every tensor it reads "
                                        "or writes once (a fused block: its input -- which is also its residual "
                                        "-- its output and its weights; the expanded tensors never reach HBM)"},
        "unfused_layers_reference": {"roof_us": round(unfused_roof_s * 1e6, 1), "bytes": tot_by, "flops": tot_fl,
                                     "note": "the same sum over the 32 convs as separate layers (expanded "
                                             "tensors written and read): bytes the fused step does not move, "
                                             "a reference only, no fraction"},
        "block_choices": model.choice_map(),
        "roofline": roofline,
        "hbm_copy_gbs": round(copy_gbs, 1),
        "cpu_baseline": cpu,
        "kernels": kernels,
    }
    print(json.dumps(out), flush=True)
    return 0


# Workloads --profile-config can run alone: (kind, n, h, w, cin, cout, stride, activation)
PROFILE_CONFIGS = {
    "pw_32to64_relu6_80x144": ("pw", 1, 80, 144, 32, 64, 1, "RELU6"),
    "pw_960to160_10x18_b1": ("pw", 1, 10, 18, 960, 160, 1, "NONE"),
    "pw_960to160_10x18_b256": ("pw", 256, 10, 18, 960, 160, 1, "NONE"),
    "igemm3x3s2_16to32_relu_160x288_b32": ("ig", 32, 160, 288, 16, 32, 2, "RELU"),
    "igemm3x3s1_32to64_relu_80x144_b32": ("ig", 32, 80, 144, 32, 64, 1, "RELU"),
    "ir_block_chain_4x_64c_40x72_b64": ("chain",),
    "encoder_160x288_b64": ("encoder",),
    "segm_r11_real_160x288_b64": ("segm",),  # the real model through the native runtime, --dtype storage
    "copy_1gib": ("copy",),  # calibration: reads and writes 1 GiB
}


def profile_config(args, torch, conv, W, Model, dev, DT) -> int:
    """--profile-config: the launches of one workload only (fp32 configs as in
    the kernel table, the encoder in --dtype with --choices), so that a
    rocprofv3 counter pass sees that workload's kernels and nothing else
    (besides torch's input fills)."""
    cfg = PROFILE_CONFIGS[args.profile_config]
    reps = args.profile_reps
    rnd = lambda nel, scale=1.0: (torch.rand(nel, device=dev) * 2 - 1) * scale
    A = conv.Activation
    if cfg[0] in ("pw", "ig"):
        _, n, h, w, cin, cout, s, act = cfg
        if cfg[0] == "pw":
            spec = conv.GemmPwSpec(m=h * w, kg=cin // 4, ng=cout // 4, act=A[act], n=n)
            m = n * h * w
            x, wt = rnd(m * cin), rnd(cin * cout, 0.05)
            run = lambda y, ws: spec.run(x, wt, b, None, y, ws)
        else:
            spec = conv.ConvIgemmSpec(ih=h, iw=w, cin=cin, cout=cout, k=3, s=s, pad=(1, 1, 1, 1), act=A[act], n=n)
            oh, ow = spec.out_hw()
            m = n * oh * ow
            x, wt = rnd(n * h * w * cin), rnd(9 * cin * cout, 0.1)
            run = lambda y, ws: spec.run([x], wt, b, None, y, ws)
        b = rnd(cout, 0.01)
        y = torch.empty(m * cout, device=dev)
        ws = torch.empty(max(spec.plan().ws_bytes // 4, 1), device=dev)
        for _ in range(reps):
            run(y, ws)
    elif cfg[0] == "chain":
        layers, meta = W.ir_chain_40x72(64)
        # --choices as the bench's block_choices (e.g. "dwpw 16x16 r4" per block), else three launches per block
        m4 = Model(layers, W.make_weights(layers, seed=1), meta["n"], meta["h"], meta["w"], meta["c"], dt=DT["f32"],
                   tune=False, choices=json.loads(args.choices) if args.choices else None)
        m4.tensors["input"].uniform_(-1, 1)
        for _ in range(reps):
            m4.infer()
    elif cfg[0] == "segm":
        from ai_engine_amd import sw

        data = open(os.path.join(ROOT, "tests", "golden", "segm_r11_160x288.sw"), "rb").read()
        m = sw.SwModel(data, n=64, dt=DT[args.dtype])
        x = (torch.rand(64, 160, 288, 3, device=dev) * 2 - 1).contiguous()
        m.upload_input("input_1", x)
        for _ in range(reps):
            m.infer()
    elif cfg[0] == "copy":
        src = torch.empty(1 << 28, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        for _ in range(reps):
            dst.copy_(src)
    else:
        layers, meta = W.mnv4_small_encoder_160x288(64)
        model = Model(layers, W.make_weights(layers, seed=0), meta["n"], meta["h"], meta["w"], 3, dt=DT[args.dtype],
                      choices=json.loads(args.choices) if args.choices else None)
        x = (torch.rand(meta["n"], meta["h"], meta["w"], 3, device=dev) * 2 - 1).contiguous()
        for _ in range(reps):
            model.upload_input(x)
            model.infer()
    torch.cuda.synchronize()
    log(f"profiled {args.profile_config}: {reps} repetitions")
    return 0


def measured_traffic(key: str):
    """HBM bytes per launch of kernel `key` as the committed rocprofv3 FETCH_SIZE /
    WRITE_SIZE summary under profiles/ reports it (calibrated against a 1 GiB
    copy in the same run), or None when no summary covers this kernel."""
    import glob
    import re

    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*hbm_traffic*.md"))):
        for line in open(path):
            m = re.match(r"traffic_bytes_per_launch (.+) = (\d+)\s*$", line)
            if m and m.group(1) == key:
                return int(m.group(2))
    return None


def kernel_key(conv, op, n, dt, dtname) -> str:
    """Name of the kernel instantiation one model op launches (as the kernel
    trace names it for the fused block; descriptive for the conv kernels)."""
    if op.kind == "stem_ir_block":
        return f"ir_wave_stem_kernel<{int(dt)}>"
    if op.kind in ("ir_block", "ir_block_head"):
        # the head joined to a block runs in the block's split kernel
        p = op.spec.plan()
        bs = op.spec.block if op.kind == "ir_block_head" else op.spec
        if p.kernel in (conv.IrKernel.WAVE, conv.IrKernel.SPLIT):
            s = bs.s
            npi = 2 if ((p.th - 1) * s + 3) * ((p.tw - 1) * s + 3) <= 64 else 5
            A = conv.Activation
            rl = "true" if int(bs.act_expand) == A.RELU and int(bs.act_dw) == A.RELU else "false"
            head = f"<{int(dt)}, {bs.cin // 16}, {npi}, {-(-bs.cout // 32)}, {rl}"
            if p.kernel == conv.IrKernel.WAVE:
                return f"ir_wave_kernel{head}>"
            return f"ir_split_kernel{head}, {'true' if p.deep else 'false'}>"
        npw = -(-(-(-p.th * p.tw // 32)) // 4)
        A = conv.Activation
        clamp = all(int(x) in (A.NONE, A.RELU, A.RELU6, A.CLAMP01)
                    for x in (bs.act_expand, bs.act_dw, bs.act_project))
        return f"ir_block_kernel<{int(dt)}, {-(-bs.cout // 32)}, {npw}, {'true' if clamp else 'false'}>"
    Lr = op.layers[0]
    if Lr.depthwise:
        return f"conv_dw_strip_kernel<{dtname}>"
    if Lr.k == 1 and -(-Lr.cout // 4) == 1:
        return f"pw_narrow_kernel<{dtname}>"
    if Lr.k == 1:
        p = conv.GemmPwSpec(m=Lr.ih * Lr.iw, kg=-(-Lr.cin // 4), ng=-(-Lr.cout // 4), dt=dt, n=n).plan()
        if p.bm == 16:
            return f"pw_splitk_kernel<{dtname}, {p.splitk}>"
        direct = f"pw_direct_kernel<{dtname}>"
    else:
        p = conv.ConvIgemmSpec(ih=Lr.ih, iw=Lr.iw, cin=Lr.cin, cout=Lr.cout, k=Lr.k, s=Lr.s, pad=(Lr.pad,) * 4,
                               dt=dt, n=n).plan()
        if p.bm == 16:
            return f"conv_ksplit_kernel<{dtname}>"
        direct = f"conv_stem_kernel<{dtname}>" if Lr.cin <= 3 else f"conv_igemm_direct_kernel<{dtname}>"
    oh, ow = Lr.out_hw()
    streamed = p.bm == 64 or (Lr.cin > 3 and p.grid == -(-n * oh * ow // 64) * -(-Lr.cout // 64))
    if streamed or p.variant == conv.Variant.DIRECT:
        return f"conv_stream_kernel<{dtname},{'igemm' if Lr.k > 1 else 'pw'}>" if streamed else direct
    key = f"conv_gemm_kernel<{dtname},{dtname},BN={p.bn},{'igemm' if Lr.k > 1 else 'pw'}>"
    return key + ("+splitk_reduce" if p.splitk > 1 else "")


def time_launches(torch, stream, fn, reps: int, warm: int = 3) -> float:
    """Median seconds of fn() measured with HIP events on the launch stream."""
    for _ in range(warm):
        fn(0)
    ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(reps)]
    for r in range(reps):
        ev[r][0].record(stream)
        fn(r)
        ev[r][1].record(stream)
    torch.cuda.synchronize()
    ts = sorted(a.elapsed_time(b) for a, b in ev)
    return ts[len(ts) // 2] / 1e3


def time_graph(torch, fn, reps: int, warm: int = 3) -> float:
    """Seconds per launch of fn(r, stream) with no host launch cost between
    kernels: reps launches (rotating buffer sets) captured once into a HIP
    graph, the graph replayed three times, the median replay / reps. Short
    kernels timed one launch at a time also measure the host's launch path
    (the Python descriptor, the plan call); this is the kernels' own rate."""
    cap = torch.cuda.Stream()
    for r in range(warm):
        fn(r, cap)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        for r in range(reps):
            fn(r, cap)
    torch.cuda.synchronize()
    cur = torch.cuda.current_stream()
    ts = []
    for _ in range(3):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record(cur)
        g.replay()
        b.record(cur)
        torch.cuda.synchronize()
        ts.append(a.elapsed_time(b) / 1e3 / reps)
    del g
    return sorted(ts)[1]


def kernel_table(torch, conv, W, Model, dev, stream, DT) -> dict:
    res = {}

    def sets_for(footprint: int) -> int:
        return max(1, math.ceil(2 * MALL_BYTES / footprint))

    def rnd(nel, dtype=torch.float32, scale=1.0):
        return (torch.rand(nel, device=dev, dtype=dtype) * 2 - 1) * scale

    def pw_case(name, n, h, w, cin, cout, act, splitk=0, reps=60):
        spec = conv.GemmPwSpec(m=h * w, kg=cin // 4, ng=cout // 4, act=act, n=n, splitk=splitk)
        plan = spec.plan()
        m = n * h * w
        fl = 2 * m * cin * cout
        by = 4 * (m * cin + cin * cout + cout + m * cout)
        S = sets_for(4 * (m * cin + m * cout))
        xs = [rnd(m * cin) for _ in range(S)]
        ys = [torch.empty(m * cout, device=dev) for _ in range(S)]
        wt = rnd(cin * cout, scale=0.05)
        b = rnd(cout, scale=0.01)
        ws = torch.empty(max(plan.ws_bytes // 4, 1), device=dev)
        t1 = time_launches(torch, stream, lambda r: spec.run(xs[r % S], wt, b, None, ys[r % S], ws, stream), reps)
        t = time_graph(torch, lambda r, st: spec.run(xs[r % S], wt, b, None, ys[r % S], ws, st), reps)
        row = roof(fl, by, t, "f32")
        row.update(us_one_launch=t1 * 1e6, variant=conv.Variant(plan.variant).name, splitk=plan.splitk, bn=plan.bn,
                   grid=plan.grid, buffer_sets=S)
        res[name] = {k: (round(v, 4) if isinstance(v, float) else v) for k, v in row.items()}
        log(f"{name}: {row['us']:.2f} us ({t1 * 1e6:.2f} us one launch at a time) {row['tflops']:.2f} TF "
            f"{row['gbs']:.0f} GB/s frac {row['frac']:.3f} {row['variant']}")

    def ig_case(name, n, ih, iw, cin, cout, s, act, reps=30):
        spec = conv.ConvIgemmSpec(ih=ih, iw=iw, cin=cin, cout=cout, k=3, s=s, pad=(1, 1, 1, 1), act=act, n=n)
        plan = spec.plan()
        oh, ow = spec.out_hw()
        m = n * oh * ow
        fl = 2 * m * 9 * cin * cout
        by = 4 * (n * ih * iw * cin + 9 * cin * cout + cout + m * cout)
        S = sets_for(4 * (n * ih * iw * cin + m * cout))
        xs = [rnd(n * ih * iw * cin) for _ in range(S)]
        ys = [torch.empty(m * cout, device=dev) for _ in range(S)]
        wt = rnd(9 * cin * cout, scale=0.1)
        b = rnd(cout, scale=0.01)
        ws = torch.empty(max(plan.ws_bytes // 4, 1), device=dev)
        t1 = time_launches(torch, stream, lambda r: spec.run([xs[r % S]], wt, b, None, ys[r % S], ws, stream), reps)
        t = time_graph(torch, lambda r, st: spec.run([xs[r % S]], wt, b, None, ys[r % S], ws, st), reps)
        row = roof(fl, by, t, "f32")
        row.update(us_one_launch=t1 * 1e6, variant=conv.Variant(plan.variant).name, splitk=plan.splitk, bn=plan.bn,
                   grid=plan.grid, buffer_sets=S)
        res[name] = {k: (round(v, 4) if isinstance(v, float) else v) for k, v in row.items()}
        log(f"{name}: {row['us']:.2f} us ({t1 * 1e6:.2f} us one launch at a time) {row['tflops']:.2f} TF "
            f"{row['gbs']:.0f} GB/s frac {row['frac']:.3f} {row['variant']}")

    # launch floor: the smallest kernel there is (a 4-byte fill) replayed back
    # to back in a graph -- what any single launch costs at the least
    tiny = torch.empty(1, device=dev)
    floor = time_graph(torch, lambda r, st: tiny.fill_(float(r)), 200)
    res["launch_floor_graph_us"] = round(floor * 1e6, 3)
    log(f"launch floor (4-byte fill, graph replay): {floor * 1e6:.2f} us")

    A = conv.Activation
    pw_case("pw_32to64_relu6_80x144", 1, 80, 144, 32, 64, A.RELU6, reps=200)
    for s in (1, 4, 8):
        pw_case(f"pw_960to160_10x18_b1_splitk{s}", 1, 10, 18, 960, 160, A.NONE, splitk=s, reps=200)
    pw_case("pw_960to160_10x18_b1_policy", 1, 10, 18, 960, 160, A.NONE, splitk=0, reps=200)
    for s in (1, 4, 8):
        pw_case(f"pw_960to160_10x18_b256_splitk{s}", 256, 10, 18, 960, 160, A.NONE, splitk=s, reps=40)
    pw_case("pw_960to160_10x18_b256", 256, 10, 18, 960, 160, A.NONE, reps=40)
    for k in ("pw_32to64_relu6_80x144", "pw_960to160_10x18_b1_policy"):
        res[k]["us_above_launch_floor"] = round(res[k]["us"] - floor * 1e6, 3)
    ig_case("igemm3x3s2_16to32_relu_160x288_b32", 32, 160, 288, 16, 32, 2, A.RELU)
    ig_case("igemm3x3s1_32to64_relu_80x144_b32", 32, 80, 144, 32, 64, 1, A.RELU)

    # four inverted-residual blocks, fp32
    layers, meta = W.ir_chain_40x72(64)
    wts = W.make_weights(layers, seed=1)
    m4 = Model(layers, wts, meta["n"], meta["h"], meta["w"], meta["c"], dt=DT["f32"])
    m4.tensors["input"].uniform_(-1, 1)
    t = time_launches(torch, stream, lambda r: m4.infer(stream), 10)
    fl = sum(op.flops(meta["n"]) for op in m4.ops)
    by = sum(op.bytes(meta["n"], 4, 4) for op in m4.ops)
    row = roof(fl, by, t, "f32")
    row["launches"] = len(m4.ops)
    row["block_choices"] = {k: {"choice": v[0], "us": round(v[1], 2)} for k, v in m4.choices.items()}
    own_s = sum(max(op.flops(meta["n"]) / (PEAK_TF["f32"] * 1e12), op.bytes(meta["n"], 4, 4) / (HBM_GBS * 1e9))
                for op in m4.ops)
    row["frac"] = own_s / t
    row["own_roofline_us"] = own_s * 1e6
    row["frac_basis"] = ("the launches' own roofline: sum over the launches run of max(flops / MFMA peak, "
                         "bytes / 8 TB/s), each launch counting every tensor it reads or writes once (the "
                         "fused depthwise + projection never writes the depthwise output); bytes and gbs "
                         "are those launches' bytes")
    row["unfused_layers_roof_us"] = sum(
        max(L.flops(meta["n"]) / (PEAK_TF["f32"] * 1e12), L.bytes(meta["n"], 4, 4) / (HBM_GBS * 1e9))
        for L in layers) * 1e6
    res["ir_block_chain_4x_64c_40x72_b64"] = {k: (round(v, 4) if isinstance(v, float) else v) for k, v in row.items()}
    log(f"ir chain: {row['us']:.1f} us frac {row['frac']:.3f}; blocks: " +
        ", ".join(f"{k} {v[0]} ({v[1]:.0f} us)" for k, v in m4.choices.items()))
    del m4
    return res


def fused_label(sw, f) -> str:
    """What a native-runtime fused block runs: its kernel plan, or the fold."""
    if f.kind == sw.FUSED_RESIZE_CONCAT:
        return "resize folded into concat"
    return str(f.dwpw if f.kind == sw.FUSED_DWPW else f.plan)


def real_model(torch, conv, dev, stream) -> dict:
    """The reference converter's real segmentation model (tests/golden/
    segm_r11_160x288.sw: 36 convs + resize / gpool / binary / concat) through
    the native .sw runtime, batch 64, fp32 as converted and with 16-bit
    storage converted at load, as loaded by default (its four inverted-
    residual blocks fused), f16 also with load-time tuning (AIH_MODEL_TUNE),
    and op by op; one step = device upload + the whole graph."""
    from ai_engine_amd import sw

    data = open(os.path.join(ROOT, "tests", "golden", "segm_r11_160x288.sw"), "rb").read()
    g, _ = sw.read_container(data)
    T = g["tensors"]
    macs = 0
    for op in g["ops"]:
        if op["kind"] == "conv":
            o = T[op["out"]]
            macs += o["h"] * o["w"] * op["kh"] * op["kw"] * op["cin"] * op["cout"] // op["groups"]
    n = 64
    x = (torch.rand(n, 160, 288, 3, device=dev) * 2 - 1).contiguous()
    out = {}
    for dt, fuse, tune in (("f32", True, False), ("f16", True, False), ("f16", True, True), ("f32", False, False),
                           ("f16", False, False)):
        m = sw.SwModel(data, n=n, dt=None if dt == "f32" else conv.DType.F16, fuse=fuse, tune=tune)

        def step(_):
            m.upload_input("input_1", x, stream)
            m.infer(stream)

        t = time_launches(torch, stream, step, 10)
        key = f"segm_r11_real_160x288_b{n}_{dt}" + ("" if fuse else "_unfused") + ("_tuned" if tune else "")
        out[key] = dict(us=round(t * 1e6, 1), frames_per_s=round(n / t, 1), tflops=round(2 * macs * n / t / 1e12, 2),
                        gflop_per_frame=round(2 * macs / 1e9, 3), ops=len(g["ops"]), launches=m.info.n_launches,
                        fused_blocks=[f"ops {f.first_op}-{f.first_op + f.n_ops - 1}: " + fused_label(sw, f)
                                      for f in m.fused_blocks()])
        log(f"real segm model {dt} b{n} {'fused' if fuse else 'unfused'}{' tuned at load' if tune else ''}: "
            f"{t * 1e3:.3f} ms {n / t:.0f} frames/s "
            f"({m.info.n_launches} launches)")
        m.close()
    return out


def encoder_native(torch, W, layers, wts, x, n, H, Wd, dt, stream, headline_fps) -> dict:
    """The headline step through the graph-level C ABI: the same encoder and
    weights written as the reference converter's .sw container, loaded by
    aih_model_load_ex with load-time tuning (AIH_MODEL_TUNE) and 16-bit
    storage. As in the headline, the input is resident before the timed
    region: uploaded once (aih_model_upload_input_device copies it into the
    model's staging buffer, which the stem then reads at every infer), and one
    step = aih_model_infer. The upload's own cost (a device-to-device copy of
    the fp32 frames) is timed apart as upload_us."""
    from ai_engine_amd import sw

    data = sw.conv_graph_to_sw("mnv4_small_encoder_160x288", layers, wts, H, Wd, 3)
    m = sw.SwModel(data, n=n, dt=dt, tune=True)
    out = m.outputs[0]

    def timed(fn, K=50):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(K):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / K

    t_up = timed(lambda: m.upload_input("input", x, stream))
    m.upload_input("input", x, stream)
    timed(lambda: m.infer(stream), 100)  # untimed: the steady state first, as for the headline
    t = timed(lambda: m.infer(stream))
    # per launch: op ranges (a fused block's ops together), HIP events around
    # each, median of 5 passes
    fb = {f.first_op: f.n_ops for f in m.fused_blocks()}
    ranges, i = [], 0
    while i < m.info.n_ops:
        ranges.append((i, i + fb.get(i, 1)))
        i += fb.get(i, 1)
    R = 5
    evs = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in ranges]
           for _ in range(R)]
    for r in range(R):
        for (a, b), (e0, e1) in zip(ranges, evs[r]):
            e0.record(stream)
            m.infer_range(a, b, stream)
            e1.record(stream)
    torch.cuda.synchronize()
    per_launch = [dict(ops=f"{a}-{b - 1}", us=round(sorted(evs[r][j][0].elapsed_time(evs[r][j][1])
                                                           for r in range(R))[R // 2] * 1e3, 2))
                  for j, (a, b) in enumerate(ranges)]
    row = dict(us=round(t * 1e6, 1), frames_per_s=round(n / t, 1), ratio_to_headline=round(n / t / headline_fps, 4),
               upload_us=round(t_up * 1e6, 1), launches=m.info.n_launches, per_launch=per_launch, output=out,
               fused_blocks=[f"ops {f.first_op}-{f.first_op + f.n_ops - 1}: {f.plan}" for f in m.fused_blocks()])
    log(f"encoder via aih_model_* ({m.info.n_launches} launches): {t * 1e3:.3f} ms {n / t:.0f} frames/s "
        f"({row['ratio_to_headline']:.3f} of the headline)")
    m.close()
    return row


def encoder_other(torch, W, Model, layers, wts, x, n, H, Wd, dtname, DT, stream) -> dict:
    m = Model(layers, wts, n, H, Wd, 3, dt=DT[dtname])

    def step(_):
        m.upload_input(x)
        m.infer()

    t = time_launches(torch, stream, step, 10)
    fl, by = W.totals(layers, n, 2, 2)
    row = roof(fl, sum(op.bytes(n, 2, 2) for op in m.ops), t, dtname)
    row["frac"] = sum(max(op.flops(n) / (PEAK_TF[dtname] * 1e12), op.bytes(n, 2, 2) / (HBM_GBS * 1e9))
                      for op in m.ops) / t
    row["frac_basis"] = ("the step's own roofline: sum over the launches run of max(flops / MFMA peak, "
                         "bytes / 8 TB/s), a fused block counting its input, output, residual and weights")
    row["unfused_layers_roof_us"] = sum(
        max(L.flops(n) / (PEAK_TF[dtname] * 1e12), L.bytes(n, 2, 2) / (HBM_GBS * 1e9)) for L in layers) * 1e6
    row["frames_per_s"] = n / t
    log(f"encoder {dtname}: {t * 1e3:.3f} ms {n / t:.0f} frames/s")
    return {k: (round(v, 4) if isinstance(v, float) else v) for k, v in row.items()}


def cpu_baseline(layers, wts, H, Wd, budget_s: float, W=None, parity_in=None) -> dict:
    """The oracle's ai-cpu restatement (the reference's CPU path) timed on the
    host's cores: the encoder (fp32, one frame at a time as ai-cpu has no
    batch, row-band threads over every core) on a bounded sample of frames --
    the reported baseline -- and every config per image at T = 1 and T = all
    cores (median of >= 3 runs after a warm-up), scaled to the config's batch.

    parity_in = (x_img0, y_img0, dtname): the GPU's input and output of image
    0 of the benchmarked batch; the same frame through the oracle gives the
    headline's parity figures (literal max |g-c|/max(|c|,1) and rms-scaled,
    each next to what ideal 16-bit storage of the same network gives)."""
    import numpy as np

    from oracle import oracle as orc

    try:
        cores = len(os.sched_getaffinity(0))
    except AttributeError:
        cores = os.cpu_count() or 1

    def chain_fn(lys, w_, rd=None):
        rd = rd or (lambda v: v)
        cc = []
        for L in lys:
            op = orc.conv2d(L.cin, L.cout, k=L.k, s=L.s, pad=L.pad, groups=L.groups, act=L.act)
            cc.append((L, orc.CpuConv(op, L.ih, L.iw, rd(w_.w[L.name]), rd(w_.b[L.name]),
                                      has_res=L.res is not None)))

        def run(x, threads):
            bufs = {"input": rd(x)}
            for L, c in cc:
                bufs[L.name] = rd(c.run(bufs[L.src], 1, bufs[L.res] if L.res else None, threads=threads))
            return bufs[lys[-1].name]
        return run

    enc = chain_fn(layers, wts)
    rng = np.random.default_rng(5)
    x = rng.uniform(-1, 1, H * Wd * 3).astype(np.float32)

    enc(x, cores)  # warm-up (also sizes the sample)
    t0 = time.perf_counter()
    enc(x, cores)
    t1 = time.perf_counter() - t0
    frames = max(2, min(4096, int(budget_s / max(t1, 1e-6))))
    t0 = time.perf_counter()
    for _ in range(frames):
        enc(x, cores)
    secs = time.perf_counter() - t0
    fps = frames / secs
    log(f"cpu baseline: {fps:.2f} frames/s on {cores} threads ({frames} frames, {secs:.1f} s)")
    out = {"value": round(fps, 3), "unit": "frames/s", "cores": cores, "kind": "port",
           "sample": f"{frames} frames of the 160x288 encoder, fp32, one frame at a time, {cores} row-band threads",
           "ms_per_frame": round(secs / frames * 1e3, 2)}

    # every config, per image, at T = 1 and T = all
    def med_time(fn, reps=3):
        fn()
        ts = []
        for _ in range(reps):
            t = time.perf_counter()
            fn()
            ts.append(time.perf_counter() - t)
        return sorted(ts)[len(ts) // 2]

    def conv_fn(cin, cout, k, s, h, w, act):
        rng_ = np.random.default_rng(cin * 1000 + cout)
        op = orc.conv2d(cin, cout, k=k, s=s, pad=(k - 1) // 2, act=act)
        cc = orc.CpuConv(op, h, w, (rng_.standard_normal(cout * cin * k * k) * 0.05).astype(np.float32),
                         (rng_.standard_normal(cout) * 0.01).astype(np.float32))
        xi = rng_.uniform(-1, 1, h * w * cin).astype(np.float32)
        return lambda T: cc.run(xi, 1, threads=T)

    rows = {}
    cfgs = [("pw_32to64_relu6_80x144", 1, conv_fn(32, 64, 1, 1, 80, 144, "relu6")),
            ("pw_960to160_10x18_b1", 1, conv_fn(960, 160, 1, 1, 10, 18, "none")),
            ("pw_960to160_10x18_b256", 256, conv_fn(960, 160, 1, 1, 10, 18, "none")),
            ("igemm3x3s2_16to32_relu_160x288_b32", 32, conv_fn(16, 32, 3, 2, 160, 288, "relu")),
            ("igemm3x3s1_32to64_relu_80x144_b32", 32, conv_fn(32, 64, 3, 1, 80, 144, "relu"))]
    if W is not None:
        c4l, c4m = W.ir_chain_40x72(64)
        c4 = chain_fn(c4l, W.make_weights(c4l, seed=1))
        x4 = rng.uniform(-1, 1, c4m["h"] * c4m["w"] * c4m["c"]).astype(np.float32)
        cfgs.append(("ir_block_chain_4x_64c_40x72_b64", 64, lambda T: c4(x4, T)))
    cfgs.append(("mnv4_small_encoder_160x288_b64", 64, lambda T: enc(x, T)))
    for name, batch, fn in cfgs:
        t_1 = med_time(lambda: fn(1))
        t_all = med_time(lambda: fn(cores))
        rows[name] = {"batch": batch, "ms_per_image_t1": round(t_1 * 1e3, 3), "ms_per_image_tall": round(t_all * 1e3, 3),
                      "ms_per_batch_t1": round(t_1 * batch * 1e3, 2), "ms_per_batch_tall": round(t_all * batch * 1e3, 2),
                      "frames_per_s_t1": round(1 / t_1, 2), "frames_per_s_tall": round(1 / t_all, 2)}
        log(f"cpu {name}: {t_1 * 1e3:.2f} ms/image T=1, {t_all * 1e3:.2f} ms/image T={cores}")
    out["per_config"] = rows
    out["per_config_protocol"] = (f"one image per run (ai-cpu has no batch; a batch is that many sequential "
                                  f"images), warm-up then median of 3, T=1 and T={cores} row-band threads")

    if parity_in is not None:
        x0, y0, dtname = parity_in
        dt = {"f16": 1, "bf16": 2}[dtname]
        ref = enc(x0, cores)
        ideal = chain_fn(layers, wts, lambda v: orc.round_to(v, dt))(x0, cores)

        def lit(g, c):
            g, c = np.asarray(g, np.float64), np.asarray(c, np.float64)
            return float(np.max(np.abs(g - c) / np.maximum(np.abs(c), 1.0)))

        def rms(g, c):
            g, c = np.asarray(g, np.float64), np.asarray(c, np.float64)
            sc = max(float(np.sqrt(np.mean(c ** 2))), 1.0)
            return float(np.max(np.abs(g - c) / np.maximum(np.abs(c), sc)))

        out["parity"] = {
            "image": 0, "against": "oracle ai-cpu chain, fp32, same frame and weights",
            "max_rel_err": round(lit(y0, ref), 5), "ideal_storage_max_rel_err": round(lit(ideal, ref), 5),
            "rms_scaled_err": round(rms(y0, ref), 5), "ideal_storage_rms_scaled_err": round(rms(ideal, ref), 5),
            "bar": 2e-2,
            "note": "He-init encoder without normalisation: activations grow to ~150 and outputs cancel, so "
                    "ideal 16-bit storage (RNE, exact fp32 arithmetic) itself misses the literal bar; "
                    "the kernels' own error is checked per launch in tests/test_gpu_workloads.py"}
        log(f"parity image 0: {out['parity']}")
    return out


if __name__ == "__main__":
    sys.exit(main())
