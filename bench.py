"""Benchmark: one Hy3 MoE FFN layer on one MI355X through libhy3x.so.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--config 0..4]
                    [--rotate N] [--secondary] [--cpu-seconds S]

A step is one forward of the MoE block (RMSNorm, router, top-8, 8 routed + 1
shared Q4_K SwiGLU experts, combine, residual) over one batch of synthetic
input already resident in HBM. The default line measures both halves of the
headline metric: decode of one token (config 0; `value`) and one 512-token
prefill chunk (config 2; the `prefill` object). The decode is timed cold:
four distinct resident layers (8.2 GB of Q4_K) are cycled one per step, so
no step finds its 99 MB of weights in the 256 MB last-level cache, as in a
real 79-layer decode (--rotate 1 re-runs one layer, cache-warm).
--secondary adds the other configurations inside the same JSON object.

Prints ONE JSON line (rank 0). Fields beyond the driver's contract:
  roofline      dominant kernel: algorithmic bytes per launch / its mean launch
                duration (HIP events on the launch stream around back-to-back
                launches of that kernel after the timed steps, rotating over the
                same resident layers); traffic = HBM bytes per launch from the
                committed rocprofv3 PMC summary
  prefill       config 2 with its own roofline (HBM and MFMA fractions)
  cpu_baseline  the reference CPU MoE block (hy3.c forward_layer_moe compiled
                from the reference sources into oracle/_ref/libhy3ref.so, built
                in the development container and shipped with the tree) or, when
                that library is absent, the oracle port, on a bounded token
                sample, with the host CPU model and the threads used
"""
import argparse
import dataclasses
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
PEAK_F16_TFLOPS = 2500.0
MAT = 3538944
Q8MAT = 7077888  # one matrix in hy3's Q8_0 (the shared expert of real checkpoints)


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=0, help="timed steps (0: per-config default)")
    p.add_argument("--warmup", type=int, default=20)
    p.add_argument("--config", type=int, default=0)
    p.add_argument("--secondary", action="store_true", help="also measure the other configs")
    p.add_argument("--cpu-seconds", type=float, default=12.0)
    p.add_argument("--rotate", type=int, default=4,
                   help="distinct resident layers a one-layer config cycles through, one per "
                        "step (4 x 2.05 GB: every step streams from HBM; 1: one layer re-run, "
                        "cache-warm at decode)")
    p.add_argument("--no-prefill", action="store_true",
                   help="skip the 512-token prefill entry (config 2) of the default line")
    p.add_argument("--no-cpu", action="store_true")
    p.add_argument("--path", type=int, default=0, choices=(0, 1, 2, 3, 4, 5),
                   help="expert path: 0 the library's choice by T, 1 GEMV tiles, 2 MFMA tiles, "
                        "3 / 4 MFMA with the narrow (32-token) / wide (64-token) tile shape, "
                        "5 MFMA with 128-token tiles")
    p.add_argument("--tokens", type=int, default=0,
                   help="override the config's token count (tuning sweeps)")
    p.add_argument("--shared-q8", action="store_true",
                   help="shared expert in hy3's Q8_0, the type real checkpoints carry "
                        "(the configs' default is Q4_K)")
    p.add_argument("--timeline", type=int, default=0, metavar="FORWARDS",
                   help="print the per-block timeline of the cold decode launches over FORWARDS "
                        "forwards (trace checkpoints) and exit")
    p.add_argument("--read-ceiling", action="store_true",
                   help="print the streaming-read rate at the decode and prefill launch sizes "
                        "(the achievable reference for the roofline fractions) and exit")
    p.add_argument("--residual", action="store_true",
                   help="time hy3x_layer_forward_residual (x += attn_out fused in front of "
                        "the block, as add_rmsnorm_kernel + gpu_ffn_moe)")
    p.add_argument("--graph", action="store_true",
                   help="replay a HIP graph of each step's kernels instead of launching them "
                        "directly (measured slower than direct launches on ROCm 7.2)")
    p.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                   help="only run a plain device copy of MIB MiB --steps times (the known-size "
                        "kernel that scales rocprofv3 FETCH_SIZE/WRITE_SIZE readings)")
    return p.parse_args()


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "pmc_traffic.json")
PEAK_MFMA_TFLOPS = 2500.0  # MI355X dense fp16 MFMA


def measured_traffic(workload, kernel):
    """HBM bytes per launch of `kernel` on `workload` from the committed rocprofv3
    --pmc FETCH_SIZE / WRITE_SIZE summary (already scaled by the copy-kernel
    calibration), or None when that kernel/workload has not been counted."""
    try:
        with open(TRAFFIC_FILE) as f:
            t = json.load(f)
        r = t["workloads"][workload][kernel]
        return int(r["fetch_bytes"] + r["write_bytes"])
    except (OSError, KeyError, ValueError):
        return None


def copy_calibration(torch, mib, steps):
    n = mib * (1 << 20) // 4
    src = torch.ones(n, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(max(steps, 1)):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration_bytes_each_way": n * 4, "launches": max(steps, 1)}))


def default_steps(T, n_layers):
    if n_layers > 1:
        return 20
    return {1: 2000, 32: 500}.get(T, 50 if T <= 512 else 10)


def stage_bytes(stage, U, T, K, decode, shared_q8=False):
    """Algorithmic HBM bytes of one launch of a kernel stage. Single-token
    decode: the router stage also streams the shared expert's gate/up and the
    gate/up stage streams the K routed experts only. shared_q8: the shared
    expert's matrices are hy3 Q8_0 (Q8MAT bytes each)."""
    sh = Q8MAT if shared_q8 else MAT
    router = 192 * 4096 * 4 + 4096 * 4 + T * 4096 * 4 + T * 4096 * 6
    if decode:
        if stage == "gateup":
            return K * 2 * MAT + 4096 * 2 + K * 1536 * 2
        if stage == "down":
            return K * MAT + sh + (K + 1) * 1536 * 2 + 2 * 4096 * 4
        if stage == "router":
            return router + 2 * sh + 1536 * 2
        return 0
    if stage == "gateup":
        return (U - 1) * 2 * MAT + 2 * sh + T * 4096 * 2 + T * (K + 1) * 1536 * 2
    if stage == "down":
        return (U - 1) * MAT + sh + T * (K + 1) * (1536 * 2 + 4096 * 4)
    if stage == "router":
        return router
    return 0


def measure(torch, H, C, cfg, steps, warmup, use_graph=False, path=0, shared_q8=False,
            residual=False, rotate=1):
    """Time `steps` forwards of cfg. A stacked config (n_layers > 1) runs all its
    layers per step. A one-layer config with rotate > 1 keeps `rotate` distinct
    layers of the same distribution resident (layer indices 0 .. rotate-1, each
    with its own scratch) and step i runs layer i % rotate: with their weights far
    beyond the 256 MB last-level cache every step streams from HBM, as the
    layers of a real decode do (cold timing). rotate = 1 re-runs one layer
    (warm for a decode, whose 99 MB stay in the cache)."""
    n_inst = cfg.n_layers if cfg.n_layers > 1 else rotate
    layers = []
    for li in range(n_inst):
        # each layer its own scratch: the stage replays below re-run a layer's
        # kernels on the routing its own last forward left there
        L = H.MoELayer(cfg.T)
        L.synth_experts(cfg.weight_seed, li)
        if shared_q8:
            L.synth_shared_q8_0(cfg.weight_seed, li)
        nw, rt, b = C.config_tensors(cfg, li)
        L.set_router(nw, rt, b)
        if path:
            L.set_path(path)
        layers.append(L)
    x = torch.from_numpy(C.inputs(cfg.input_seed, cfg.T).copy()).cuda()
    # residual addend (attention output stand-in): a small multiple of other inputs
    attn = torch.from_numpy(C.inputs(cfg.input_seed + 1, cfg.T).copy() * 0.01).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    stacked = cfg.n_layers > 1
    turn = [0]

    def fwd(L, st=stream):
        if residual:
            L.forward_residual(x.data_ptr(), attn.data_ptr(), cfg.T, cfg.K, stream=st)
        else:
            L.forward(x.data_ptr(), cfg.T, cfg.K, stream=st)

    def eager_step():
        if stacked:
            for L in layers:
                fwd(L)
        else:
            fwd(layers[turn[0] % n_inst])
            turn[0] += 1

    step = eager_step
    if use_graph:
        # one graph per step (a stacked config: every layer's kernels), replayed as one launch
        assert stacked or n_inst == 1, "--graph times one layer or a stack"
        eager_step()
        torch.cuda.synchronize()
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            with torch.cuda.graph(graph, stream=side):
                for L in layers:
                    fwd(L, side.cuda_stream)
        torch.cuda.current_stream().wait_stream(side)
        step = graph.replay

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    for L in layers:
        L.stats(reset=True)
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    fw, touched = zip(*[L.stats(reset=True) for L in layers])
    U = sum(touched) / max(sum(fw), 1)  # mean experts touched per layer-forward
    ms = elapsed * 1e3 / steps
    tokens_per_s = cfg.T * steps / elapsed

    # per-stage timing pass (HIP events on the launch stream)
    for L in layers:
        L.set_timing(True)
    for _ in range(steps):
        eager_step()
    torch.cuda.synchronize()
    stages = {}
    nfw = 0
    for L in layers:
        st, n = L.stage_times()
        nfw += n
        for k, v in st.items():
            stages[k] = stages.get(k, 0.0) + v
        L.set_timing(False)
    stage_us = {k: v * 1e3 / max(nfw, 1) for k, v in stages.items()}
    dom = max(("gateup", "down"), key=lambda k: stage_us[k])
    kernel = layers[0].last_kernel(dom)
    decode = cfg.T == 1 and layers[0].path == 0
    dom_bytes = stage_bytes(dom, U, cfg.T, cfg.K, decode, shared_q8)
    # launch duration of the dominant kernel: replayed back to back on the launch
    # stream between two HIP events, after the timed forwards
    reps = max(10, min(steps, 2000))
    launch_us = H.layers_time_stage(layers, dom, reps, stream=stream)
    achieved = dom_bytes / (launch_us * 1e-6) / 1e9
    # the kernel's binding roofline: its arithmetic intensity against the
    # machine balance (2.5 PFLOP/s dense fp16 MFMA over 8 TB/s = 312 flop/B)
    per_slot = (4 if dom == "gateup" else 2) * 1536 * 4096  # flop per (token, expert)
    dom_flops = 0 if decode else per_slot * cfg.T * (cfg.K + 1)
    tflops = dom_flops / (launch_us * 1e-6) / 1e12
    mfma_bound = dom_flops / dom_bytes > PEAK_MFMA_TFLOPS * 1e12 / (PEAK_HBM_GBS * 1e9)
    alg_bytes = (C.algorithmic_bytes(cfg.T, U) + (3 * (Q8MAT - MAT) if shared_q8 else 0)) * cfg.n_layers
    flops = C.algorithmic_flops(cfg.T, cfg.K) * cfg.n_layers
    for L in layers:
        L.close()
    return dict(
        tokens_per_s=tokens_per_s, ms_per_step=ms, U=U, layer_GBps=alg_bytes / (ms * 1e-3) / 1e9,
        layer_TFLOPs=flops / (ms * 1e-3) / 1e12, stage_us=stage_us,
        roofline=(dict(bound="mfma", kernel=kernel, achieved=round(tflops, 1),
                       peak=PEAK_MFMA_TFLOPS, unit="TFLOP/s",
                       frac=round(tflops / PEAK_MFMA_TFLOPS, 4),
                       hbm_GBps=round(achieved, 1), hbm_frac=round(achieved / PEAK_HBM_GBS, 4))
                  if mfma_bound else
                  dict(bound="hbm", kernel=kernel, achieved=round(achieved, 1), peak=PEAK_HBM_GBS,
                       unit="GB/s", frac=round(achieved / PEAK_HBM_GBS, 4),
                       **({} if decode else dict(mfma_TFLOPs=round(tflops, 1),
                                                 mfma_frac=round(tflops / PEAK_MFMA_TFLOPS, 4)))))
        | dict(traffic=measured_traffic(f"config{cfg.index}:{cfg.name}", kernel),
               bytes_per_launch=int(dom_bytes), flops_per_launch=int(dom_flops),
               launch_us=round(launch_us, 3),
               launch_timing=f"HIP events around {reps} back-to-back launches over "
                             f"{len(layers)} resident layer(s) in rotation"),
    )


def cpu_model():
    """The host CPU's model name (from /proc/cpuinfo), or the platform string."""
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    import platform
    return platform.processor() or platform.machine()


def cpu_baseline(torch, H, C, cfg, seconds, shared_q8=False):
    """hy3.c's CPU MoE block on a bounded token sample (same Q4_K bytes; with
    shared_q8 the same Q8_0 shared expert)."""
    from oracle import hy3_oracle as O
    from hy3_amd import hipmem
    L = H.MoELayer(1)
    L.synth_experts(cfg.weight_seed, 0)
    lay = O.SynthLayer(cfg.weight_seed, 0,
                       zipf_seed=cfg.input_seed if cfg.zipf_bias else None, shared_q8=shared_q8)
    for e in range(193 if not shared_q8 else 192):
        lay.experts[e] = tuple(hipmem.to_host(L.expert_ptr(e, m), MAT) for m in range(3))
    L.close()
    ref = O.ref_lib()
    kind = "reference" if ref is not None else "port"
    if ref is None:
        # oracle/_ref is built from the reference sources in the development
        # container and travels with the working tree; a clean checkout lacks it
        print(f"bench.py: WARNING: {O.REF_LIB} is absent; cpu_baseline times the oracle port "
              "(kind 'port'), not hy3.c's own forward_layer_moe", file=sys.stderr, flush=True)
        ref_build = None
    else:
        import hashlib
        with open(O.REF_LIB, "rb") as f:
            ref_build = {"library": os.path.relpath(O.REF_LIB, ROOT),
                         "sha256": hashlib.sha256(f.read()).hexdigest()}
    cores = os.cpu_count() or 1
    cores = min(cores, int(os.environ.get("OMP_NUM_THREADS", cores)))
    if ref is not None:
        ref.hy3ref_set_threads(cores)
    else:
        O.lib().hy3o_set_num_threads(cores)
    n, t0 = 0, time.perf_counter()
    while True:
        x = C.inputs(cfg.input_seed, 1, first_token=n)
        if ref is not None:
            lay.ref_forward(x, cfg.K)
        else:
            lay.forward(x, cfg.K)
        n += 1
        el = time.perf_counter() - t0
        if el >= seconds or n >= 100000:
            break
    return dict(value=round(n / el, 3), unit="tokens/s", cores=cores, kind=kind,
                reference_build=ref_build, cpu_model=cpu_model(),
                prefill_note="hy3.c runs a prefill's MoE one token at a time (hy3_gpu.cu:836-837, "
                             "hy3.c per-token forward), so its prefill tokens/s equals this rate",
                sample=f"{n} tokens of config {cfg.index}, one at a time as hy3.c runs its MoE "
                       f"(forward_layer_moe per token), {el:.1f} s")


def decode_timeline(torch, forwards):
    """Per-block timeline of the cold single-token decode (config 0, four
    resident layers in rotation): every block of the three launches writes
    REALTIME-counter checkpoints (hy3x_layer_set_trace; 100 MHz); prints, per
    checkpoint, the median over forwards of the blocks' median / 90th
    percentile / last time in us from the first route block's start."""
    import numpy as np
    import hy3_amd as H
    from hy3_amd import configs as C
    torch.cuda.init()
    cfg = C.CONFIGS[0]
    layers = []
    for li in range(4):
        L = H.MoELayer(1)
        L.synth_experts(cfg.weight_seed, li)
        nw, rt, b = C.config_tensors(cfg, li)
        L.set_router(nw, rt, b)
        layers.append(L)
    x = torch.from_numpy(C.inputs(cfg.input_seed, 1).copy()).cuda()
    # trace buffers: 8 checkpoints per block; stage 0 384 blocks (192 router,
    # 192 of shared rows), stage 1 K x 384 routed gate/up blocks, stage 2 256
    # down (sized with room to spare; blocks that did not run stay zero and
    # are dropped)
    bufs = [torch.zeros(n * 8, dtype=torch.int64, device="cuda") for n in (1024, 8192, 1024)]
    for i in range(50):
        layers[i % 4].forward(x.data_ptr(), 1)
    torch.cuda.synchronize()
    rows = []
    for i in range(10 + forwards):
        L = layers[i % 4]
        for st, bf in enumerate(bufs):
            bf.zero_()
            H._check(H.lib().hy3x_layer_set_trace(L._h, st, bf.data_ptr()))
        torch.cuda.synchronize()
        L.forward(x.data_ptr(), 1)
        torch.cuda.synchronize()
        for st in range(3):
            H._check(H.lib().hy3x_layer_set_trace(L._h, st, None))
        if i < 10:
            continue
        r, g, d = (bf.cpu().numpy().reshape(-1, 8).astype(np.float64) for bf in bufs)
        r, g, d = (a[a[:, 0] > 0] for a in (r, g, d))
        t0 = r[:, 0].min()
        us = lambda v: (v - t0) / 100.0
        rows.append({
            "route: block start": us(r[:, 0]),
            "route: router x/row loaded": us(r[:192, 1]),
            "route: router chains done": us(r[:192, 3]),
            "route: shared s staged": us(r[192:, 1]),
            "route: shared rows done": us(r[192:, 3]),
            "gate/up: block start": us(g[:, 0]),
            "gate/up: routed, s staged": us(g[:, 1]),
            "gate/up: rows done": us(g[:, 3]),
            "down: block start": us(d[:, 0]),
            "down: rows done": us(d[:, 2]),
            "down: combine written": us(d[:, 3])})
    out = []
    for k in rows[0]:
        out.append({"checkpoint": k,
                    "median_us": round(float(np.median([np.median(r[k]) for r in rows])), 2),
                    "p90_us": round(float(np.median([np.percentile(r[k], 90) for r in rows])), 2),
                    "last_us": round(float(np.median([r[k].max() for r in rows])), 2)})
    print(json.dumps({"decode_timeline": out, "forwards": forwards,
                      "timing": "cold: 4 resident layers in rotation"}), flush=True)


def main():
    a = parse()
    if a.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {a.gpus}); "
              "multi-GPU sharding (expert or tensor parallel) is not implemented.", file=sys.stderr)
        sys.exit(2)
    import torch
    if a.copy_calibration:
        copy_calibration(torch, a.copy_calibration, a.steps)
        return
    if a.timeline:
        decode_timeline(torch, a.timeline)
        return
    if a.read_ceiling:
        import hy3_amd as H
        torch.cuda.init()
        pool = torch.empty(4 << 30, dtype=torch.uint8, device="cuda").fill_(1)
        rows = []
        for mb in (8, 16, 32, 56, 96, 256, 1024):
            us = H.read_rate_us(pool.data_ptr(), pool.numel(), mb << 20)
            rows.append({"MiB": mb, "us": round(us, 2), "GB_per_s": round((mb << 20) / us / 1e3, 1)})
        print(json.dumps({"read_ceiling": rows, "pool": "4 GiB, rotating slots"}), flush=True)
        return
    import hy3_amd as H
    from hy3_amd import configs as C
    torch.cuda.init()
    cfg = C.CONFIGS[a.config]
    if a.tokens:
        cfg = dataclasses.replace(cfg, T=a.tokens, name=f"{cfg.name}@T{a.tokens}")
    steps = a.steps or default_steps(cfg.T, cfg.n_layers)
    rotate = a.rotate if cfg.n_layers == 1 else 1
    r = measure(torch, H, C, cfg, steps, a.warmup, use_graph=a.graph, path=a.path,
                shared_q8=a.shared_q8, residual=a.residual, rotate=rotate)
    out = {
        "metric": "MoE-layer tokens/s at decode B=1 and 512-tok prefill; achieved HBM GB/s vs peak",
        "value": round(r["tokens_per_s"], 2),
        "unit": "tokens/s",
        "n_gpus": 1, "steps": steps, "warmup": a.warmup,
        "ms_per_step": round(r["ms_per_step"], 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "q4k-weights/fp16-act/fp32-acc",
        "data": "synthetic (seeded, BASELINE configs; random-init Q4_K weights)",
        "config": {"workload": f"config{cfg.index}:{cfg.name}", "tokens": cfg.T,
                   "layers": cfg.n_layers, "top_k": cfg.K, "experts": "192+1 shared",
                   "hidden": 4096, "ffn": 1536, "parallelism": "single-gpu",
                   "timing": (f"cold: {rotate} resident layers "
                              f"({rotate * 2.05:.1f} GB of Q4_K) in rotation, one per step"
                              if rotate > 1 else
                              "stack: every layer per step" if cfg.n_layers > 1 else
                              "one layer re-run every step"),
                   "launch": "hip-graph" if a.graph else "direct",
                   "expert_path": ["auto", "gemv", "mfma", "mfma-narrow", "mfma-wide", "mfma-big"][a.path],
                   "shared_expert": "q8_0" if a.shared_q8 else "q4_k",
                   "entry": "forward_residual" if a.residual else "forward"},
        "layer": {"experts_touched": round(r["U"], 2), "GB_per_s": round(r["layer_GBps"], 1),
                  "hbm_frac": round(r["layer_GBps"] / PEAK_HBM_GBS, 4),
                  "stage_us": {k: round(v, 2) for k, v in r["stage_us"].items()}},
        "roofline": r["roofline"],
    }
    if cfg.index == 0 and not a.no_prefill and not a.tokens:
        # the metric's second half: one 512-token prefill chunk (config 2)
        c2 = C.CONFIGS[2]
        steps2 = default_steps(c2.T, 1)
        rp = measure(torch, H, C, c2, steps2, 5, path=a.path, shared_q8=a.shared_q8)
        out["prefill"] = {
            "workload": f"config{c2.index}:{c2.name}", "tokens": c2.T, "steps": steps2,
            "tokens_per_s": round(rp["tokens_per_s"], 1),
            "ms_per_step": round(rp["ms_per_step"], 4),
            "experts_touched": round(rp["U"], 1),
            "GB_per_s": round(rp["layer_GBps"], 1),
            "hbm_frac": round(rp["layer_GBps"] / PEAK_HBM_GBS, 4),
            "TFLOP_per_s": round(rp["layer_TFLOPs"], 2),
            "mfma_frac": round(rp["layer_TFLOPs"] / PEAK_MFMA_TFLOPS, 4),
            "stage_us": {k: round(v, 1) for k, v in rp["stage_us"].items()},
            "roofline": rp["roofline"]}
        torch.cuda.empty_cache()
    if a.secondary:
        sec = {}
        for c in C.CONFIGS:
            if c.index == cfg.index:
                continue
            rr = measure(torch, H, C, c, default_steps(c.T, c.n_layers), 3,
                         use_graph=a.graph, shared_q8=a.shared_q8)
            sec[f"config{c.index}:{c.name}"] = {
                "tokens_per_s": round(rr["tokens_per_s"], 1),
                "ms_per_step": round(rr["ms_per_step"], 4),
                "GB_per_s": round(rr["layer_GBps"], 1), "TFLOP_per_s": round(rr["layer_TFLOPs"], 2),
                "experts_touched": round(rr["U"], 1),
                "stage_us": {k: round(v, 1) for k, v in rr["stage_us"].items()},
                "roofline": rr["roofline"]}
            torch.cuda.empty_cache()
        out["secondary"] = sec
    if not a.no_cpu:
        out["cpu_baseline"] = cpu_baseline(torch, H, C, cfg, a.cpu_seconds, a.shared_q8)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
