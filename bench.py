#!/usr/bin/env python3
"""Benchmark of the quantized-SDPA hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload 2] [--skip-cpu-baseline]

A step is one pass of the whole path (K statistics, INT8 Q/K quantization, V repack,
attention, bf16 output) over one synthetic batch that is already resident in
HBM.  The workload is the Flux/Klein joint text+image attention shape
B=1, H=24, S=4608, D=128 (INT8 QK^T, FP16 PV).  One JSON line is printed:

  value          effective attention TOPS = 4*B*H*S^2*D / step time
  roofline       the attention kernel alone (the dominant kernel), timed with
                 HIP events on the launch stream, against the dense INT8 MFMA peak
  cpu_baseline   the CPU checker's implementation of the same path, timed on
                 this machine's host cores (a reported baseline, not a target)

  roofline.traffic  HBM bytes per launch of that kernel as measured with rocprofv3 --pmc
                 (FETCH_SIZE, WRITE_SIZE), read from the summary under profiles/ that
                 `--summarize-traffic` wrote; null when the kernel's source has changed since

This path runs on a single GPU; --gpus above 1 is refused.

    python bench.py --summarize-traffic FETCH_DIR WRITE_DIR FETCH_COPY_DIR WRITE_COPY_DIR
        turns the four rocprofv3 --pmc output directories (attention kernel and the 256 MiB
        calibration copy, one counter each) into the text of profiles/<kernel>_hbm_traffic.txt
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

METRIC = "effective attention TOPS at H=24,S=4608,D=128; % of INT8/FP8 MFMA peak"
PEAK_INT8_TOPS = 5000.0      # MI355X dense INT8 MFMA, published
PEAK_FP8_TOPS = 5000.0       # MI355X dense FP8 MFMA, published
PEAK_HBM_GBS = 8000.0
K_FLAGS = 3                  # K mean smoothing + per-channel Q/K balancing (the default recipe)

KERNEL_SOURCE = "mojodiffusion_amd/csrc/sage_attn.hip"
KERNEL_HEADER = "mojodiffusion_amd/csrc/sage_internal.h"


def kernel_source_digest():
    """Digest of what the attention kernel is compiled from: its source file and, of the shared
    header, the tile constants and the argument struct it uses (the other kernels' structs in
    that header do not change it)."""
    import hashlib
    import re
    h = hashlib.sha256()
    with open(os.path.join(ROOT, KERNEL_SOURCE), "rb") as f:
        h.update(f.read())
    with open(os.path.join(ROOT, KERNEL_HEADER)) as f:
        text = f.read()
    for line in text.split("\n"):
        if line.startswith("constexpr int k"):
            h.update(line.encode())
    for name in ("struct KeyMask", "struct AttnArgs", "inline int v_slot_f16", "inline int v_slot_fp8"):
        m = re.search(re.escape(name) + r".*?\n}", text, re.S)
        assert m is not None, name
        h.update(m.group(0).encode())
    return h.hexdigest()[:16]


def traffic_summary_path(workload_name):
    return os.path.join(ROOT, "profiles", "attention_%s_hbm_traffic.txt" % workload_name)


def measured_traffic(workload_name):
    """HBM bytes per launch of the attention kernel from the committed counter summary, or None
    when there is none for this workload or the kernel's source has changed since it was taken."""
    path = traffic_summary_path(workload_name)
    if not os.path.exists(path):
        return None
    kv = {}
    for line in open(path):
        if "=" in line and not line.lstrip().startswith("#"):
            k, v = line.split("=", 1)
            kv[k.strip()] = v.strip()
    if kv.get("kernel_source_digest") != kernel_source_digest():
        return None
    return int(kv["traffic_bytes_per_launch"])


def summarize_traffic(dirs):
    """rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE report KiB per dispatch.  The same counters on a
    plain 256 MiB device copy (which reads and writes exactly 256 MiB) give the scale factors."""
    import csv
    import glob

    def avg(d, pattern):
        f = glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True)
        vals = [float(r["Counter_Value"]) for r in csv.DictReader(open(f[0])) if pattern in r["Kernel_Name"]]
        # the copy kernel is the one whose value is largest (torch launches helpers too)
        return sum(vals) / len(vals), len(vals)

    def copy_avg(d):
        f = glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True)
        by = {}
        for r in csv.DictReader(open(f[0])):
            by.setdefault(r["Kernel_Name"], []).append(float(r["Counter_Value"]))
        name = max(by, key=lambda k: sum(by[k]) / len(by[k]))
        return sum(by[name]) / len(by[name]), name
    fetch, n_f = avg(dirs[0], "sage_attn_kernel")
    write, n_w = avg(dirs[1], "sage_attn_kernel")
    fetch_copy, cname = copy_avg(dirs[2])
    write_copy, _ = copy_avg(dirs[3])
    copy_kib = 256.0 * 1024.0
    f_scale, w_scale = copy_kib / fetch_copy, copy_kib / write_copy
    total = int(round((fetch * f_scale + write * w_scale) * 1024.0))
    print("# HBM traffic of sage_attn_kernel per launch, rocprofv3 --pmc (one counter per run)")
    print("# Commands (repository root on the MI355X box, after `cd /tmp && export TMPDIR=/tmp` and back; OUT = any "
          "scratch directory), C = FETCH_SIZE, then WRITE_SIZE:")
    print("#   rocprofv3 --pmc C --output-format csv -d OUT/pmc_C_bench -o p -- python3 bench.py --skip-cpu-baseline --skip-other-workloads --steps 3 --warmup 2")
    print("#   rocprofv3 --pmc C --output-format csv -d OUT/pmc_C_copy -o p -- python3 bench.py --copy-calibration")
    print("#   python3 bench.py --summarize-traffic OUT/pmc_FETCH_SIZE_bench OUT/pmc_WRITE_SIZE_bench "
          "OUT/pmc_FETCH_SIZE_copy OUT/pmc_WRITE_SIZE_copy")
    print("kernel_source_digest = %s" % kernel_source_digest())
    print("fetch_size_kib_per_dispatch = %.1f   # %d dispatches" % (fetch, n_f))
    print("write_size_kib_per_dispatch = %.1f   # %d dispatches" % (write, n_w))
    print("copy_kernel = %s" % cname.split("(")[0][:80])
    print("copy_fetch_size_kib = %.1f   # for 262144 KiB read: scale %.4f" % (fetch_copy, f_scale))
    print("copy_write_size_kib = %.1f   # for 262144 KiB written: scale %.4f" % (write_copy, w_scale))
    print("traffic_bytes_per_launch = %d" % total)



def clock_probe(args, L, w, qd, kd, vd, o, st, stream):
    """The chip lowers its shader clock under this kernel (power management).  The measurement
    build's attention kernel stamps s_memtime (shader clocks) and s_memrealtime (100 MHz) at its
    start and end; their ratio is the clock each workgroup ran at."""
    import numpy as np
    import torch
    from mojodiffusion_amd import _lib
    P = ctypes.CDLL(args.probe_lib or os.path.join(os.path.dirname(_lib.LIB_PATH), "libmi355_sage_probe.so"))
    for name in ("mi355_sage_quant_qk_bf16", "mi355_sage_quant_v_f16", "mi355_sage_quant_v_fp8", "mi355_sage_attn_fwd"):
        getattr(P, name).restype, getattr(P, name).argtypes = _lib.SIGNATURES[name]
    assert P.mi355_sage_set_attn_split(-1) == 0     # the main kernel, which stamps, for the whole problem (the short form does not)
    B, S, H, D = w.B, w.S, w.H, w.D
    dev = qd.device
    nqp, nkp = L.mi355_sage_pad_q(S), L.mi355_sage_pad_kv(S)
    q8 = torch.empty((B, H, nqp, D), dtype=torch.int8, device=dev)
    k8 = torch.empty((B, H, nkp, D), dtype=torch.int8, device=dev)
    qs = torch.empty((B, H, nqp // w.blkq), dtype=torch.float32, device=dev)
    ks = torch.empty((B, H, nkp // w.blkk), dtype=torch.float32, device=dev)
    km, qm, kmu, vsc = (torch.empty((B, H, D), dtype=torch.float32, device=dev) for _ in range(4))
    vq = torch.empty((B, H, nkp // 64, D, 64), dtype=torch.int16 if w.variant == 0 else torch.uint8, device=dev)
    scr = torch.empty(max(L.mi355_sage_quant_scratch_bytes(B, H, S, D), 8), dtype=torch.uint8, device=dev)
    nwg = (nqp // 256) * B * H
    stats = torch.zeros(B * H * S + 2 * nwg, dtype=torch.float32, device=dev)      # Stats, then the stamps
    assert P.mi355_sage_quant_qk_bf16(qd.data_ptr(), kd.data_ptr(), B, H, S, S, D, w.scale, st, st, 0, 0, w.blkq, w.blkk,
                                      K_FLAGS, 0, 0, q8.data_ptr(), qs.data_ptr(), k8.data_ptr(), ks.data_ptr(),
                                      km.data_ptr(), qm.data_ptr(), kmu.data_ptr(), scr.data_ptr(), scr.numel(), stream) == 0
    if w.variant == 0:
        assert P.mi355_sage_quant_v_f16(vd.data_ptr(), B, H, S, D, st, 0, 0, 0, vq.data_ptr(), stream) == 0
    else:
        assert P.mi355_sage_quant_v_fp8(vd.data_ptr(), B, H, S, D, st, 0, 0, 0, vq.data_ptr(), vsc.data_ptr(),
                                        scr.data_ptr(), scr.numel(), stream) == 0

    def attn():
        assert P.mi355_sage_attn_fwd(q8.data_ptr(), qs.data_ptr(), w.blkq, k8.data_ptr(), ks.data_ptr(), w.blkk,
                                     vq.data_ptr(), vsc.data_ptr(), w.variant, B, H, S, S, S, 0, 0, D,
                                     o.data_ptr(), st, 0, None, stats.data_ptr(), stream) == 0
    for _ in range(args.warmup + args.steps):               # back to back, as in a sampler's layer loop
        attn()
    torch.cuda.synchronize()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    attn()
    b.record()
    torch.cuda.synchronize()
    x = stats[B * H * S:].cpu().numpy().reshape(nwg, 2).astype(np.float64)
    mhz = x[:, 0] / x[:, 1] * 100.0
    tiles = (S + 63) // 64
    per_xcd = [round(float(np.median(mhz[i::8])), 1) for i in range(8)]     # consecutive workgroups go to the 8 XCDs in turn
    print(json.dumps({
        "workload": w.name, "kernel_ms": round(a.elapsed_time(b), 5), "workgroups": nwg,
        "shader_clock_mhz": {"mean": round(float(mhz.mean()), 1), "median": round(float(np.median(mhz)), 1),
                             "p10": round(float(np.quantile(mhz, 0.1)), 1), "p90": round(float(np.quantile(mhz, 0.9)), 1)},
        "median_shader_clock_mhz_per_xcd": per_xcd,
        "shader_clocks_per_workgroup": round(float(x[:, 0].mean()), 0),
        "shader_clocks_per_64_key_tile": round(float(x[:, 0].mean()) / tiles, 1),
        "matrix_pipe_clocks_per_tile_per_simd": 2 * (8 * 32 + (16 * 32 if w.variant == 0 else 4 * 64)),
    }))


def run_workload(L, torch, w, qd, kd, vd, steps, warmup, n_events):
    """One workload through the one-shot call (wall clock over back-to-back steps) and through the
    stage entry points with HIP events on the launch stream, each stage as the one-shot call runs it:
    the quantize stage (one launch by hand-over, mi355_sage_quant_once, where the call makes that; otherwise the
    launches of mi355_sage_quant_qkv_bf16, which calls under capture make too) and the attention kernel.  Where the
    one-shot call leaves the Q encode to the attention kernel (every shape but those of the split
    schedule), so do the stages timed here: the quantize stage without Q outputs and mi355_sage_attn_fwd_q16."""
    from mojodiffusion_amd import _lib
    dev = qd.device
    B, S, H, D = w.B, w.S, w.H, w.D
    o = torch.empty_like(qd)
    st = _lib.strides_bhnd(S, H, D)
    nws = L.mi355_sage_workspace_bytes(B, H, S, S, D, w.variant)
    ws = torch.empty(nws, dtype=torch.uint8, device=dev)
    stream = torch.cuda.current_stream().cuda_stream

    def step(on_stream=stream):
        rc = L.mi355_sage_sdpa_bf16_ex(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), o.data_ptr(),
                                       B, H, S, S, D, w.scale, st, st, st, st, 0, 0, 0, 0, 0, on_stream,
                                       w.variant, w.blkq, w.blkk, K_FLAGS, ws.data_ptr(), nws)
        if rc != 0:
            raise RuntimeError("mi355_sage_sdpa_bf16_ex rc=%d" % rc)

    # The chip takes some milliseconds of load to leave its idle clocks (a 50-step run right after
    # start-up reads 12 % slower than a 1000-step one): run the same step, untimed, for 0.15 s
    # before the warm-up proper, whatever --warmup says.
    ramp_steps = 0
    r0 = time.perf_counter()
    while time.perf_counter() - r0 < 0.15:
        for _ in range(4):
            step()
        torch.cuda.synchronize()
        ramp_steps += 4
    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / steps

    nqp, nkp = L.mi355_sage_pad_q(S), L.mi355_sage_pad_kv(S)
    q8 = torch.empty((B, H, nqp, D), dtype=torch.int8, device=dev)
    k8 = torch.empty((B, H, nkp, D), dtype=torch.int8, device=dev)
    qs = torch.empty((B, H, nqp // w.blkq), dtype=torch.float32, device=dev)
    ks = torch.empty((B, H, nkp // w.blkk), dtype=torch.float32, device=dev)
    km, qm, kmu, vsc = (torch.empty((B, H, D), dtype=torch.float32, device=dev) for _ in range(4))
    vq = torch.empty((B, H, nkp // 64, D, 64), dtype=torch.int16 if w.variant == 0 else torch.uint8, device=dev)
    # (and the hand-over's flags: 16 bytes per head and group of 256 keys)
    scr = torch.empty(L.mi355_sage_quant_scratch_bytes(B, H, S, D) + 16 * B * H * ((S + 255) // 256), dtype=torch.uint8, device=dev)

    def stage_quant(with_q, once=False):
        outs = (q8.data_ptr() if with_q else None, qs.data_ptr() if with_q else None, k8.data_ptr(), ks.data_ptr(), km.data_ptr(),
                qm.data_ptr(), kmu.data_ptr(), vq.data_ptr(), vsc.data_ptr(), scr.data_ptr(), scr.numel())
        x = (qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), B, H, S, S, D, w.scale, st, st, st)
        if once:                              # (64 looks: the one-shot call's own)
            return L.mi355_sage_quant_once(*x, w.variant, w.blkq, 0, 0, None, None, 0.0, None, None, 0, *outs, 64, stream)
        return L.mi355_sage_quant_qkv_bf16(*x, 0, 0, 0, w.variant, w.blkq, w.blkk, K_FLAGS, 0, 0, *outs, stream)

    def attn_q8():
        return L.mi355_sage_attn_fwd(q8.data_ptr(), qs.data_ptr(), w.blkq, k8.data_ptr(), ks.data_ptr(), w.blkk,
                                     vq.data_ptr(), vsc.data_ptr(), w.variant, B, H, S, S, S, 0, 0, D,
                                     o.data_ptr(), st, 0, None, None, stream)

    def attn_q16():
        return L.mi355_sage_attn_fwd_q16(qd.data_ptr(), st, 0, qm.data_ptr(), w.blkq, k8.data_ptr(), ks.data_ptr(), w.blkk,
                                         vq.data_ptr(), vsc.data_ptr(), w.variant, B, H, S, S, S, 0, 0, D,
                                         o.data_ptr(), st, 0, stream)

    assert stage_quant(True) == 0
    rc = attn_q16()                       # -2: a shape of the split schedule, whose Q the quantize stage encodes
    if rc not in (0, -2):
        raise RuntimeError("mi355_sage_attn_fwd_q16 rc=%d" % rc)
    q_in_kernel = rc == 0
    stage_attn = attn_q16 if q_in_kernel else attn_q8

    def time_stage(fn, n):
        for _ in range(3):
            assert fn() == 0
        torch.cuda.synchronize()
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]
        for a, b in evs:
            a.record()
            assert fn() == 0
            b.record()
        torch.cuda.synchronize()
        ts = sorted(a.elapsed_time(b) for a, b in evs)
        return sum(ts) / len(ts), ts[len(ts) // 2], ts[0]

    once = L.mi355_sage_quant_once_takes(B, H, S, S, D, w.variant, w.blkq, w.blkk, K_FLAGS, not q_in_kernel) == 1
    qt_avg, qt_med, qt_min = time_stage(lambda: stage_quant(not q_in_kernel, once), n_events)
    at_avg, at_med, at_min = time_stage(stage_attn, n_events)
    return dict(step=step, ms_per_step=ms_per_step, ramp_steps=ramp_steps, quant=(qt_avg, qt_med, qt_min),
                attn=(at_avg, at_med, at_min), q_in_kernel=q_in_kernel, once=once, keep=(o, ws, q8, k8, qs, ks, km, qm, kmu, vsc, vq, scr))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--workload", type=int, default=2)
    ap.add_argument("--skip-cpu-baseline", action="store_true")
    ap.add_argument("--skip-other-workloads", action="store_true",
                    help="leave out config.other_workloads (the other DiT shapes, a few steps each)")
    ap.add_argument("--summarize-traffic", nargs=4, metavar="DIR",
                    help="print the traffic summary from four rocprofv3 --pmc output directories (no GPU needed)")
    ap.add_argument("--clock-probe", action="store_true",
                    help="run the attention kernel of a measurement build (default libmi355_sage_probe.so), which records "
                         "its own shader cycles and elapsed constant-rate time per workgroup, and print the clock "
                         "the chip sustained under it and the shader clocks a 64-key tile took")
    ap.add_argument("--probe-lib", default=None, help="measurement build --clock-probe loads (a path)")
    ap.add_argument("--probe-heads", type=int, default=None,
                    help="--clock-probe with this many heads instead of the workload's (few heads: a cool, idle chip)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a plain device copy of 256 MiB (read 256 MiB, write 256 MiB) five times: "
                         "the known-size kernel the HBM traffic counters are scaled by")
    args = ap.parse_args()
    if args.summarize_traffic:
        summarize_traffic(args.summarize_traffic)
        return
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this hot path is measured on ONE GPU (heads are independent and would shard "
              "without any exchange); run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch

    from mojodiffusion_amd import _lib
    from mojodiffusion_amd.workloads import WORKLOADS, make_inputs, device_inputs

    if not torch.cuda.is_available():
        print("bench.py: no GPU visible; the library has no CPU path", file=sys.stderr)
        sys.exit(3)
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.copy_calibration:
        src = torch.full((256 << 20,), 7, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_each_way": src.numel(), "launches": 5}))
        return
    L = _lib.lib()
    w = WORKLOADS[args.workload]
    if args.clock_probe and args.probe_heads:
        w = w.scaled(H=args.probe_heads)
    q, k, v = make_inputs(w)
    up = lambda x: torch.from_numpy(x.view(np.int16)).to(dev).view(torch.bfloat16)
    qd, kd, vd = up(q), up(k), up(v)
    B, S, H, D = w.B, w.S, w.H, w.D
    st = _lib.strides_bhnd(S, H, D)
    stream = torch.cuda.current_stream().cuda_stream

    if args.clock_probe:
        clock_probe(args, L, w, qd, kd, vd, torch.empty_like(qd), st, stream)
        return

    n_ev = max(args.steps, 20)
    r = run_workload(L, torch, w, qd, kd, vd, args.steps, args.warmup, n_ev)
    ms_per_step = r["ms_per_step"]
    tops = w.ops / (ms_per_step * 1e-3) / 1e12

    # ---- the same step replayed from a HIP graph: what a caller that captures its layer loop sees.
    # 200 replays after 50, whatever --steps says (a handful of replays mostly measures the ramp).
    graph_ms = None
    try:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            cap_stream = torch.cuda.current_stream().cuda_stream
            with torch.cuda.graph(g, stream=side):
                r["step"](cap_stream)
            for _ in range(50):
                g.replay()
            torch.cuda.synchronize()
            g0 = time.perf_counter()
            for _ in range(200):
                g.replay()
            torch.cuda.synchronize()
            graph_ms = (time.perf_counter() - g0) * 1e3 / 200
    except Exception as e:                                  # reported, never fatal for the headline number
        print("bench.py: graph replay timing skipped: %r" % (e,), file=sys.stderr)
    torch.cuda.synchronize()

    qt_avg, qt_med, qt_min = r["quant"]
    at_avg, at_med, at_min = r["attn"]
    attn_tops = w.ops / (at_avg * 1e-3) / 1e12
    peak = PEAK_INT8_TOPS if w.variant == 0 else PEAK_FP8_TOPS
    # algorithmic HBM bytes of the quantize stage: K and V (and Q, where this stage encodes it) read once
    # as bf16; int8 K (and Q) and fp16 / e4m3 V written
    elems = B * H * S * D
    fused = r["q_in_kernel"]
    vbytes = 2 if w.variant == 0 else 1
    quant_bytes = (2 if fused else 3) * elems * 2 + (1 if fused else 2) * elems + elems * vbytes
    quant_gbs = quant_bytes / (qt_avg * 1e-3) / 1e9

    out = {
        "metric": METRIC,
        "value": round(tops, 2),
        "unit": "TOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8/f16" if w.variant == 0 else "int8/f8e4m3",
        "data": "synthetic",
        "config": {
            "workload": w.name,
            "B": B, "H": H, "S": S, "D": D,
            "recipe": "K mean-smoothed, Q/K channel-balanced; Q int8 per %d tokens; K int8 per %d tokens; PV %s" % (
                w.blkq, w.blkk, "fp16" if w.variant == 0 else "fp8-e4m3 with per-channel V scales"),
            "ops_per_step": w.ops,
            "pct_of_peak": round(100.0 * tops / peak, 2),
            "peak_tops_used": peak,
            # HIP-event pairs on the launch stream around the quantize stage as the step runs it and around the attention launch
            "stage_ms": {"quantize": round(qt_avg, 5), "attn": round(at_avg, 5)},
            "q_encoded_by": "attention kernel (prologue)" if fused else "quantize stage",
            "graph_replay_ms": None if graph_ms is None else round(graph_ms, 5),
            "graph_replays": 200,
            "clock_ramp_steps": r["ramp_steps"],      # untimed steps run before the warm-up, see run_workload
            "device": torch.cuda.get_device_name(0),
        },
        "roofline": {
            "kernel": "sage_attn_kernel<%d,%d%s>" % (D, w.variant, ", Q encoded in the prologue" if fused else ""),
            "bound": "mfma",
            "achieved": round(attn_tops, 2),
            "peak": peak,
            "unit": "TFLOP/s",
            "frac": round(attn_tops / peak, 4),
            "traffic": measured_traffic(w.name),
            # Q (bf16, or int8 where the quantize stage encodes it) and int8 K read once, V^T tiles (fp16 or
            # e4m3) read once, bf16 O written once
            "algorithmic_bytes_per_launch": (2 if fused else 1) * elems + elems + elems * vbytes + 2 * elems,
            "avg_ms": round(at_avg, 5), "median_ms": round(at_med, 5), "min_ms": round(at_min, 5),
            "algorithmic_ops_per_launch": w.ops,
        },
        # the HBM-bound part of the step
        "roofline_quantize": {
            "kernels": ("quant_once_kernel (one launch)" if r["once"] else
                        "prep_kernel + stats_final_kernel + quant_kernel (one event pair around the launches)") + ("; K and V only" if fused else ""),
            "bound": "hbm",
            "achieved": round(quant_gbs, 1),
            "peak": PEAK_HBM_GBS,
            "unit": "GB/s",
            "frac": round(quant_gbs / PEAK_HBM_GBS, 4),
            "algorithmic_bytes": quant_bytes,
            "avg_ms": round(qt_avg, 5), "median_ms": round(qt_med, 5), "min_ms": round(qt_min, 5),
        },
    }
    del r

    if not args.skip_other_workloads and args.workload == 2:
        # The other DiT shapes at full size with inputs drawn on the device: a few timed steps each.
        others = {}
        plan = {3: (40, 10), 4: (12, 4), 5: (5, 2)}
        for wid, (n_steps, n_warm) in plan.items():
            ww = WORKLOADS[wid]
            qq, kk, vv = device_inputs(ww, 7000 + wid)
            rr = run_workload(L, torch, ww, qq, kk, vv, n_steps, n_warm, max(n_steps // 2, 5))
            pk = PEAK_INT8_TOPS if ww.variant == 0 else PEAK_FP8_TOPS
            t_ = ww.ops / (rr["ms_per_step"] * 1e-3) / 1e12
            a_ = ww.ops / (rr["attn"][0] * 1e-3) / 1e12
            others[ww.name] = {"steps": n_steps, "warmup": n_warm, "ms_per_step": round(rr["ms_per_step"], 4),
                               "TOPS": round(t_, 1), "pct_of_peak": round(100.0 * t_ / pk, 2),
                               "attn_kernel_avg_ms": round(rr["attn"][0], 4), "attn_kernel_frac_of_peak": round(a_ / pk, 4),
                               "quantize_avg_ms": round(rr["quant"][0], 4), "q_in_attention_kernel": rr["q_in_kernel"], "dtype": "int8/f16" if ww.variant == 0 else "int8/f8e4m3"}
            del rr, qq, kk, vv
            torch.cuda.empty_cache()
        out["config"]["other_workloads"] = others

    if not args.skip_cpu_baseline:
        from oracle import sage_oracle
        # bounded sample: whole passes over a subset of heads at the full sequence length, repeated
        # until about ten seconds of CPU work have been timed
        heads = min(H, 8)
        qh, kh, vh = (np.ascontiguousarray(x[:, :, :heads]) for x in (q, k, v))
        sage_oracle.sdpa_bf16(qh[:, :256], kh[:, :256], vh[:, :256], w.scale, w.variant, w.blkq, w.blkk)   # warm
        passes, c0 = 0, time.perf_counter()
        while True:
            sage_oracle.sdpa_bf16(qh, kh, vh, w.scale, variant=w.variant, blkq=w.blkq, blkk=w.blkk)
            passes += 1
            c1 = time.perf_counter()
            if c1 - c0 >= 10.0 or passes >= 64:
                break
        sample_ops = 4 * B * heads * S * S * D * passes
        out["cpu_baseline"] = {
            "value": round(sample_ops / (c1 - c0) / 1e12, 5),
            "unit": "TOPS",
            "cores": sage_oracle.num_threads(),
            "kind": "port",
            "sample": "%d of %d heads of the same workload at full S=%d, %d passes, %.2f s (C + OpenMP restatement; "
                      "the reference's own path is Mojo/cuDNN and cannot run here)" % (heads, H, S, passes, c1 - c0),
        }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
