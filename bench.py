#!/usr/bin/env python3
"""Benchmark of the causal-attention hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--T 4096] [--mode bf16|fp32]
                    [--workload flash_fwd|flash_bwd|ragged_fwd|layer_fwd|layer_train]

Default workload (one "step" = one dt_flash_attn_fwd launch over one batch):
causal attention at the OLMo-2-1B head shape, B=1, T=4096, H=16, D=128, bf16
Q/K/V/O with fp32 accumulation, Q/K/V ~ N(0,1) from seeds 1001-1003, already
resident in HBM. Prints one JSON line: causal-attention TFLOP/s over the
algorithmic work 2*B*H*D*T*(T+1) (unmasked pairs only, QK^T and PV, 2 flops
per MAC), the tokens/s of the attention core, the roofline fraction of the
MFMA peak, per-launch statistics, the peak re-derived from this device, and
the CPU baseline: the oracle's restatement of the reference's
flash_attention_forward (FlashAttention.cpp:24-182) timed on this host. The
default line also carries the same workload in fp32 exact mode ("fp32_exact")
and the end-to-end OLMo-2-1B prefill at T=2048 ("prefill",
"prefill_tok_per_s"); --no-extras skips those two.

Before the warm-up, every workload runs a clock-settle phase of about 100 ms
of back-to-back launches ("clock_settle" in the line): the shader clock of an
idle MI355X takes 30-50 ms of load to reach its sustained value.

Other workloads (each prints one line of the same shape):
  flash_bwd    one dt_flash_attn_bwd (FlashAttention.cpp:185-359) at the same
               shape; work 5*B*H*D*T*(T+1) (S, dP, dV, dQ, dK over unmasked pairs)
  ragged_fwd   a right-padded batch B=8, lengths U[64, 2048] (seed 4001), H=16;
               work sum_b 2*H*D*L_b*(L_b+1)
  layer_fwd    OlmoAttention::forward (OlmoAttention.cpp:56-108), x [1, T, 2048]
               (seed 2001, T=512 by default), seeded weights; work
               8*T*d^2 (q/k/v/o projections) + 2*H*D*T*(T+1)
  layer_train  forward with saved state + OlmoAttention::backward + step at the
               same shape; work 3x the projections' and 3.5x the attention
               core's forward work
  model_fwd    OlmoModel::forward end to end (OlmoModel.cpp:25-48): 16 layers,
               d_model 2048, MLP 8192, vocab 100352, tokens [1, 2048] (seed
               5001); work 16*(8*T*d^2 + 6*T*d*8192 + attention) + 2*T*d*V
  model_train  main.cpp's step for one batch: forward, ce_loss and its
               gradient, OlmoModel::backward, step
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

# MI355X dense MFMA peak (AMD's published figure); an fp32 exact product takes six bf16 ones (the fp32 instruction's
# own peak is 157.3)
PEAK_TFLOPS = {"bf16": 2500.0, "fp32": 2500.0 / 6}
FLOP_PER_CLK_PER_CU = {"bf16": 4096, "fp32": 4096 / 6}  # dense MFMA rate of one gfx950 compute unit
SCALE = 0.08838834764831845  # 1/sqrt(128) as fp32 (OlmoAttention.cpp:91)
SETTLE_MS = 100.0  # clock-settle phase: back-to-back launches before the warm-up (see main)
ORACLE_FLAGS = "-O3 -march=x86-64-v3 -ffast-math -fno-finite-math-only"  # oracle/Makefile (the reference: -ffast-math)


def algorithmic_flops(B: int, T: int, H: int, D: int) -> int:
    return 2 * B * H * D * T * (T + 1)


def cpu_model() -> str:
    try:
        for ln in open("/proc/cpuinfo"):
            if ln.startswith("model name"):
                return ln.split(":", 1)[1].strip()
    except OSError:  # pragma: no cover
        pass
    return "unknown"


def cpu_baseline(T: int, H: int, D: int, budget_s: float = 10.0) -> dict:
    """Times the oracle (the CPU restatement of FlashAttention.cpp:24-182) on the full workload,
    repeated until ``budget_s`` has passed (at least 2 runs), threads = min(B*H, usable cores) like the
    reference's TBB loop over (b, h); then on one thread over 2 of the 16 heads (the per-head work is
    identical, so the full single-thread time is 8x that), also median of repeated runs."""
    import numpy as np

    import oracle
    from dirktensor_amd import synth

    Q, K, V = synth.qkv(1, T, H)
    threads, cores = _threads(H)
    med, n = _time_cpu(lambda: oracle.flash_attention_forward(Q, K, V, SCALE, True, nthreads=threads), budget_s)
    hs = 2
    Q1, K1, V1 = (np.ascontiguousarray(x[:, :, :hs]) for x in (Q, K, V))
    med1, n1 = _time_cpu(lambda: oracle.flash_attention_forward(Q1, K1, V1, SCALE, True, nthreads=1),
                         max(budget_s / 2, 1.0))
    return {
        "value": algorithmic_flops(1, T, H, D) / med / 1e12,
        "unit": "TFLOP/s",
        "cores": threads,
        "kind": "port",
        "sample": f"oracle flash_attention_forward fp32, B=1 T={T} H={H} D={D} causal, full workload x "
                  f"{n} runs (median {med * 1e3:.1f} ms), {threads} threads of {cores} usable",
        "cpu_model": cpu_model(),
        "compile_flags": ORACLE_FLAGS,
        "fast_math": True,
        "one_thread": {"value": algorithmic_flops(1, T, hs, D) / med1 / 1e12, "unit": "TFLOP/s",
                       "sample": f"{hs} of {H} heads x {n1} runs (median {med1 * 1e3:.1f} ms) on 1 thread"},
    }


def device_peak(mode: str) -> dict:
    """The MFMA peak re-derived from this device: compute units x dense MFMA flop per clock per CU x the
    maximum shader clock that rocminfo reports for the gfx950 agent (published: 256 CUs, 2400 MHz)."""
    import subprocess

    cus, mhz, src = 256, 2400, "published (256 CUs, 2400 MHz)"
    try:
        out = subprocess.run(["rocminfo"], capture_output=True, text=True, timeout=20).stdout
        for agent in out.split("Agent ")[1:]:
            if "gfx950" not in agent:
                continue
            c = [int(ln.split(":")[1]) for ln in agent.splitlines() if ln.strip().startswith("Compute Unit:")]
            f = [int(ln.split(":")[1]) for ln in agent.splitlines() if ln.strip().startswith("Max Clock Freq. (MHz):")]
            if c and f:
                cus, mhz, src = c[0], f[0], "rocminfo"
            break
    except Exception:  # noqa: BLE001 - the published figures stand in
        pass
    peak = cus * FLOP_PER_CLK_PER_CU[mode] * mhz * 1e6 / 1e12
    return {"cus": cus, "max_sclk_mhz": mhz, "flop_per_clk_per_cu": FLOP_PER_CLK_PER_CU[mode],
            "peak_tflops": round(peak, 1), "source": src}


def load_traffic(mode: str, T: int):
    """HBM bytes per launch from the committed rocprofv3 --pmc summary of this workload, when one
    exists: the line ``traffic_bytes_per_launch: N`` of profiles/flash_fwd_<mode>_t<T>_pmc.md."""
    import re

    p = ROOT / "profiles" / f"flash_fwd_{mode}_t{T}_pmc.md"
    if not p.exists():
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*(\d+)\s*$", p.read_text(), flags=re.M)
    return int(m.group(1)) if m else None


def copy_calibration(mib: int, steps: int, warmup: int) -> int:
    """Times torch.neg over ``mib`` MiB of bf16 (reads mib MiB, writes mib MiB per launch). Profiled
    with rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE, it gives the factor between those counters and
    the bytes a kernel really moves to and from HBM."""
    import torch

    n = mib * (1 << 20) // 2
    src = torch.randn(n, device="cuda:0").to(torch.bfloat16)
    dst = torch.empty_like(src)
    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        torch.neg(src, out=dst)
    torch.cuda.synchronize()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record(stream)
    for _ in range(steps):
        torch.neg(src, out=dst)
    ev1.record(stream)
    torch.cuda.synchronize()
    ms = ev0.elapsed_time(ev1) / steps
    nbytes = 2 * mib * (1 << 20)
    print(json.dumps({"metric": "copy calibration", "bytes_per_launch": nbytes, "read_bytes": nbytes // 2,
                      "write_bytes": nbytes // 2, "ms_per_launch": round(ms, 5),
                      "GB_per_s": round(nbytes / (ms * 1e-3) / 1e9, 1)}), flush=True)
    return 0


def _events(n):
    import torch

    return [torch.cuda.Event(enable_timing=True) for _ in range(n)]


def settle_clock(step, stream, target_ms: float = SETTLE_MS) -> dict:
    """Clock-settle phase, run before the warm-up whatever --warmup says. The MI355X shader clock ramps from
    about 1.6 GHz to about 2.0 GHz over the first 30-50 ms of sustained load (measured in-kernel with s_memtime
    against s_memrealtime), so back-to-back launches totalling ``target_ms`` of GPU time put the warm-up and
    the timed region at the clock a sustained workload runs at. Reported as its own key, next to warmup."""
    import torch

    e0, e1 = _events(2)
    launches, gpu_ms, batch = 0, 0.0, 5
    while gpu_ms < target_ms and launches < 20000:
        e0.record(stream)
        for _ in range(batch):
            step()
        e1.record(stream)
        torch.cuda.synchronize()
        t = e0.elapsed_time(e1)
        launches += batch
        gpu_ms += t
        # the next batch covers what remains (at least one launch), at the rate just measured
        batch = int(min(max((target_ms - gpu_ms) / max(t / batch, 1e-3), 1), 20000 - launches)) or 1
    return {"launches": launches, "gpu_ms": round(gpu_ms, 2)}


def time_steps(step, stream, steps: int) -> tuple:
    """ms per step over ``steps`` back-to-back steps, HIP events on the launch stream; and the wall time."""
    import torch

    torch.cuda.synchronize()
    e0, e1 = _events(2)
    wall0 = time.perf_counter()
    e0.record(stream)
    for _ in range(steps):
        step()
    e1.record(stream)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / steps, time.perf_counter() - wall0


def launch_stats(step, stream, n: int, flops: float) -> dict:
    """Per-launch durations from an event pair around each of ``n`` launches (a separate pass after the timed
    region, so the events do not perturb it): median, min and p90 in microseconds, TFLOP/s at the median."""
    import numpy as np
    import torch

    ev = _events(n + 1)
    ev[0].record(stream)
    for i in range(n):
        step()
        ev[i + 1].record(stream)
    torch.cuda.synchronize()
    us = np.array([ev[i].elapsed_time(ev[i + 1]) * 1e3 for i in range(n)])
    med = float(np.median(us))
    return {"n": n, "median_us": round(med, 2), "min_us": round(float(us.min()), 2),
            "p90_us": round(float(np.percentile(us, 90)), 2), "median_tflops": round(flops / (med * 1e-6) / 1e12, 1)}


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--T", type=int, default=4096)
    ap.add_argument("--H", type=int, default=16,
                    help="heads (flash_fwd / flash_bwd; 2 is one GPU's share of 16 heads split 8 ways)")
    ap.add_argument("--mode", choices=["bf16", "fp32"], default="bf16")
    ap.add_argument("--workload", choices=["flash_fwd", "flash_bwd", "ragged_fwd", "layer_fwd", "layer_train",
                                           "model_fwd", "model_train"], default="flash_fwd")
    ap.add_argument("--cpu-budget", type=float, default=10.0, help="seconds of CPU-baseline timing (0 = skip)")
    ap.add_argument("--no-extras", action="store_true",
                    help="default workload only: skip the fp32 exact-mode and end-to-end prefill figures")
    ap.add_argument("--qkv", choices=["auto", "fused", "gemm"], default="auto",
                    help="layer/model forwards: fused QKV projection + q/k norm + RoPE kernel, the library GEMM "
                    "followed by the separate norm + RoPE kernel, or auto (fused where its tiles fit one round)")
    ap.add_argument("--gemm-tune", type=int, choices=[0, 1], default=1,
                    help="bf16 GEMMs: time hipBLASLt's heuristic candidates once per shape (1) or take its first choice (0)")
    ap.add_argument("--bwd-dq", choices=["auto", "from_ds", "recompute"], default="auto",
                    help="attention backward: dQ from the dS the dK/dV pass stores, recomputed S and dP, or "
                    "auto (the dS path with more than one 128-row block per CU and pass)")
    ap.add_argument("--side-stream", type=int, choices=[0, 1], default=1,
                    help="model backward: weight-gradient GEMMs and norm-weight column sums on a second stream beside "
                    "the input-gradient chain (1) or everything on one stream (0)")
    ap.add_argument("--copy-mib", type=int, default=0,
                    help="instead of attention, time a plain copy kernel over this many MiB (counter calibration)")
    args = ap.parse_args()

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU: the attention path is built and measured on a single MI355X "
              "(multi-GPU sharding is a design note, not part of this build). Run with --gpus 1.",
              file=sys.stderr)
        return 2

    import torch

    if args.copy_mib > 0:
        return copy_calibration(args.copy_mib, args.steps, args.warmup)

    import dirktensor_amd as dt

    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream(dev)
    ctx = dt.default_context(0)
    ctx.set_qkv_path(args.qkv)
    ctx.set_gemm_tune(bool(args.gemm_tune))
    ctx.set_bwd_dq_path(args.bwd_dq)
    ctx.set_side_stream(bool(args.side_stream))
    wl = WORKLOADS[args.workload](args, dev, stream, ctx)

    settle = settle_clock(wl["step"], stream)
    for _ in range(args.warmup):
        wl["step"]()
    # the timed region: exactly --steps steps, synchronised on both sides, events on the launch stream
    ms, wall = time_steps(wl["step"], stream, args.steps)
    stats = launch_stats(wl["step"], stream, max(args.steps, 50), wl["flops"]) if wl.get("stats", True) else None

    tflops = wl["flops"] / (ms * 1e-3) / 1e12
    peak = PEAK_TFLOPS[args.mode]
    parity = wl["parity"]()
    cpu = wl["cpu"](args.cpu_budget) if args.cpu_budget > 0 else None
    line = {
        "metric": wl["metric"],
        "value": round(tflops, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "clock_settle": settle,
        "ms_per_step": round(ms, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": args.mode,
        "data": wl["data"],
        "config": wl["config"],
        "tok_per_s": round(wl["tokens"] / (ms * 1e-3), 1),
        "pct_of_peak": round(100.0 * tflops / peak, 2),
        "parity_rel_err": parity,
        "wall_s_timed_region": round(wall, 4),
        "stats": stats,
        "peak_derivation": device_peak(args.mode),
        "roofline": {"bound": "mfma", "achieved": round(tflops, 3), "peak": peak, "unit": "TFLOP/s",
                     "frac": round(tflops / peak, 4), "traffic": wl.get("traffic")},
        "cpu_baseline": cpu,
    }
    if args.workload.startswith(("layer", "model")):
        line["config"]["gemm_choice"] = "tuned hipBLASLt candidates" if args.gemm_tune else "first hipBLASLt heuristic"
        line["config"]["qkv_projection"] = {"fused": "fused kernel", "gemm": "library GEMM + norm/RoPE kernel",
                                            "auto": "auto (fused kernel when its tiles fit one round)"}[args.qkv]
    if args.workload == "flash_fwd":
        line["attn_core_tok_per_s"] = line["tok_per_s"]  # tokens/s of the attention core alone, not prefill
    if args.workload == "model_fwd":
        line["prefill_tok_per_s"] = line["tok_per_s"]
    if args.workload == "flash_fwd" and args.mode == "bf16" and args.H == 16 and not args.no_extras:
        line["fp32_exact"] = _extra(lambda: extra_fp32_exact(args, dev, stream, ctx))
        line["prefill"] = _extra(lambda: extra_prefill(args, dev, stream, ctx))
        if isinstance(line["prefill"], dict) and "prefill_tok_per_s" in line["prefill"]:
            line["prefill_tok_per_s"] = line["prefill"]["prefill_tok_per_s"]
    print(json.dumps(line), flush=True)
    return 0


def _extra(fn):
    """An extra figure of the default line; a failure is reported in its place, not raised."""
    try:
        return fn()
    except Exception as e:  # noqa: BLE001
        return {"error": f"{type(e).__name__}: {e}"}


def extra_fp32_exact(args, dev, stream, ctx) -> dict:
    """The reference's own precision: the same attention workload in fp32 exact mode, timed like
    the headline, with its parity against the oracle on two heads. The clock is settled again first: the CPU
    baseline before it leaves the GPU idle for seconds."""
    a = argparse.Namespace(**{**vars(args), "mode": "fp32"})
    wl = wl_flash_fwd(a, dev, stream, ctx)
    settle_clock(wl["step"], stream)
    for _ in range(5):
        wl["step"]()
    steps = 20
    ms, _ = time_steps(wl["step"], stream, steps)
    tf = wl["flops"] / (ms * 1e-3) / 1e12
    return {"value": round(tf, 2), "unit": "TFLOP/s", "steps": steps, "ms_per_step": round(ms, 4),
            "pct_of_fp32_peak": round(100.0 * tf / PEAK_TFLOPS["fp32"], 2),
            "peak": round(PEAK_TFLOPS["fp32"], 1), "parity_rel_err": wl["parity"](), "tolerance": 1e-4,
            "config": wl["config"]["workload"]}


def extra_prefill(args, dev, stream, ctx) -> dict:
    """End-to-end prefill (OlmoModel::forward, OlmoModel.cpp:25-48) at the OLMo-2-1B shape, tokens [1, 2048],
    bf16 mode, weights drawn on the device: tokens/s over the whole forward (embedding to logits), with the
    logits' parity against the oracle's fp32 forward."""
    import gc

    a = argparse.Namespace(**{**vars(args), "T": 2048, "mode": "bf16"})
    wl = wl_model_fwd(a, dev, stream, ctx)
    settle_clock(wl["step"], stream)
    for _ in range(3):
        wl["step"]()
    steps = 10
    ms, _ = time_steps(wl["step"], stream, steps)
    T = wl["config"]["T"]
    out = {"prefill_tok_per_s": round(T / (ms * 1e-3), 1), "ms_per_forward": round(ms, 3), "steps": steps,
           "tflops": round(wl["flops"] / (ms * 1e-3) / 1e12, 1), "parity_rel_err": wl["parity"](),
           "tolerance": 2e-2, "config": wl["config"]["workload"] + ", 16 layers, d_model 2048, MLP 8192, vocab 100352"}
    wl["release"]()
    gc.collect()
    return out


def _threads(limit: int) -> tuple:
    try:
        cores = len(os.sched_getaffinity(0))
    except AttributeError:  # pragma: no cover
        cores = os.cpu_count() or 1
    return max(1, min(limit, cores, 16)), cores


def _time_cpu(fn, budget_s: float):
    import numpy as np

    times = []
    t_start = time.perf_counter()
    while len(times) < 2 or (time.perf_counter() - t_start < budget_s and len(times) < 50):
        t0 = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t0)
    return float(np.median(times)), len(times)


def _rel(a, b) -> float:
    import numpy as np

    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def wl_flash_fwd(args, dev, stream, ctx):
    import torch

    from dirktensor_amd import _capi, synth

    B, T, H, D = 1, args.T, args.H, 128
    tdt = torch.bfloat16 if args.mode == "bf16" else torch.float32
    dtype = _capi.DT_BF16 if args.mode == "bf16" else _capi.DT_FP32_EXACT
    Qn, Kn, Vn = synth.qkv(B, T, H)
    q, k, v = (torch.from_numpy(x).to(dev).to(tdt) for x in (Qn, Kn, Vn))
    o = torch.empty_like(q)
    m = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    l = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    fn = _capi.lib().dt_flash_attn_fwd
    args_c = (ctx.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), m.data_ptr(), l.data_ptr(),
              B, T, H, D, SCALE, 1, None, dtype, _capi.DT_MEM_DEVICE, stream.cuda_stream)

    def step():
        rc = fn(*args_c)
        if rc != 0:
            _capi.check(rc)

    def parity():  # the measured output on two heads against the oracle (fp32 inputs)
        import oracle

        O_ref, _, _ = oracle.flash_attention_forward(Qn[:, :, :2], Kn[:, :, :2], Vn[:, :, :2], SCALE, True)
        return _rel(o[:, :, :2].float().cpu().numpy(), O_ref)

    return dict(step=step, flops=algorithmic_flops(B, T, H, D), tokens=B * T, parity=parity,
                cpu=lambda budget: cpu_baseline(T, H, D, budget),
                metric="causal attn TFLOP/s + prefill tok/s, OLMo-2-1B shape T=4096 (% of MFMA peak)",
                data="synthetic (Q/K/V ~ N(0,1), seeds 1001-1003)",
                config={"workload": f"causal flash attention forward, B={B} T={T} H={H} D={D}, {args.mode}",
                        "B": B, "T": T, "H": H, "D": D, "causal": True},
                traffic=load_traffic(args.mode, T))


def wl_flash_bwd(args, dev, stream, ctx):
    import numpy as np
    import torch

    import oracle
    from dirktensor_amd import _capi, synth

    B, T, H, D = 1, args.T, args.H, 128
    tdt = torch.bfloat16 if args.mode == "bf16" else torch.float32
    dtype = _capi.DT_BF16 if args.mode == "bf16" else _capi.DT_FP32_EXACT
    Qn, Kn, Vn = synth.qkv(B, T, H)
    Gn = synth.normal(1004, Qn.shape)
    q, k, v, g = (torch.from_numpy(x).to(dev).to(tdt) for x in (Qn, Kn, Vn, Gn))
    o = torch.empty_like(q)
    m = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    l = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    _capi.call("dt_flash_attn_fwd", ctx.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
               m.data_ptr(), l.data_ptr(), B, T, H, D, SCALE, 1, None, dtype, _capi.DT_MEM_DEVICE,
               stream.cuda_stream)
    dq, dk, dv = (torch.empty_like(q) for _ in range(3))
    fn = _capi.lib().dt_flash_attn_bwd
    args_c = (ctx.handle, g.data_ptr(), o.data_ptr(), m.data_ptr(), l.data_ptr(), q.data_ptr(), k.data_ptr(),
              v.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, T, H, D, SCALE, 1, dtype,
              _capi.DT_MEM_DEVICE, stream.cuda_stream)

    def step():
        rc = fn(*args_c)
        if rc != 0:
            _capi.check(rc)

    def parity():  # two heads against the oracle's backward from the same (device) forward statistics
        hs = slice(0, 2)
        to = lambda t: t[:, :, hs].float().cpu().numpy()
        ref = oracle.flash_attention_backward(to(g), to(o), to(m), to(l), to(q), to(k), to(v), SCALE, True)
        return max(_rel(to(x), r) for x, r in zip((dq, dk, dv), ref))

    def cpu(budget):
        O, mm, ll = oracle.flash_attention_forward(Qn, Kn, Vn, SCALE, True)
        threads, cores = _threads(H)
        med, n = _time_cpu(lambda: oracle.flash_attention_backward(Gn, O, mm, ll, Qn, Kn, Vn, SCALE, True,
                                                                   nthreads=threads), budget)
        return {"value": 2.5 * algorithmic_flops(B, T, H, D) / med / 1e12, "unit": "TFLOP/s", "cores": threads,
                "kind": "port", "sample": f"oracle flash_attention_backward fp32, B=1 T={T} H={H} D={D} causal, "
                f"full workload x {n} runs (median {med * 1e3:.1f} ms), {threads} threads of {cores} usable"}

    return dict(step=step, flops=5 * B * H * D * T * (T + 1), tokens=B * T, parity=parity, cpu=cpu,
                metric=f"causal attn backward TFLOP/s, OLMo-2-1B shape T={T} (% of MFMA peak)",
                data="synthetic (Q/K/V ~ N(0,1) seeds 1001-1003, dO ~ N(0,1) seed 1004)",
                config={"workload": f"causal flash attention backward, B={B} T={T} H={H} D={D}, {args.mode}",
                        "B": B, "T": T, "H": H, "D": D, "causal": True, "dq_path": args.bwd_dq})


def wl_ragged_fwd(args, dev, stream, ctx):
    import numpy as np
    import torch

    import oracle
    from dirktensor_amd import _capi, synth

    lens = synth.ragged_lengths()
    B, H, D = len(lens), 16, 128
    T = int(lens.max())
    tdt = torch.bfloat16 if args.mode == "bf16" else torch.float32
    dtype = _capi.DT_BF16 if args.mode == "bf16" else _capi.DT_FP32_EXACT
    Qn, Kn, Vn = synth.qkv(B, T, H)
    q, k, v = (torch.from_numpy(x).to(dev).to(tdt) for x in (Qn, Kn, Vn))
    o = torch.empty_like(q)
    m = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    l = torch.empty((B, T, H), dtype=torch.float32, device=dev)
    lens_c = np.ascontiguousarray(lens, dtype=np.int32)
    fn = _capi.lib().dt_flash_attn_fwd
    args_c = (ctx.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), m.data_ptr(), l.data_ptr(),
              B, T, H, D, SCALE, 1, lens_c.ctypes.data, dtype, _capi.DT_MEM_DEVICE, stream.cuda_stream)

    def step():
        rc = fn(*args_c)
        if rc != 0:
            _capi.check(rc)

    flops = sum(2 * H * D * int(L) * (int(L) + 1) for L in lens)

    def parity():  # the shortest and the longest sequence, two heads each
        err = 0.0
        for b in (int(np.argmin(lens)), int(np.argmax(lens))):
            L = int(lens[b])
            O_ref, _, _ = oracle.flash_attention_forward(Qn[b:b + 1, :L, :2], Kn[b:b + 1, :L, :2],
                                                         Vn[b:b + 1, :L, :2], SCALE, True)
            err = max(err, _rel(o[b:b + 1, :L, :2].float().cpu().numpy(), O_ref))
        return err

    def cpu(budget):
        threads, cores = _threads(H)
        med, n = _time_cpu(lambda: oracle.flash_attention_ragged(Qn, Kn, Vn, lens, SCALE, nthreads=threads), budget)
        return {"value": flops / med / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
                "sample": f"oracle flash_attention_forward per sequence, B={B} ragged lengths {int(lens.min())}.."
                f"{T} (seed 4001), x {n} runs (median {med * 1e3:.1f} ms), {threads} threads of {cores} usable"}

    return dict(step=step, flops=flops, tokens=int(lens.sum()), parity=parity, cpu=cpu,
                metric="ragged causal attn TFLOP/s, B=8 lengths U[64,2048] (% of MFMA peak)",
                data="synthetic (Q/K/V ~ N(0,1) seeds 1001-1003, lengths seed 4001)",
                config={"workload": f"causal flash attention forward, right-padded batch B={B} T={T} H={H} "
                        f"D={D}, {args.mode}", "B": B, "T": T, "H": H, "D": D, "lengths": [int(x) for x in lens]})


def _layer_setup(args, dev):
    import torch

    from dirktensor_amd import OlmoAttention, synth

    T = args.T if args.T != 4096 else 512  # the layer workload is quoted at T = 512
    w = synth.attention_layer_weights()
    layer = OlmoAttention.from_weights(w["wq"], w["wk"], w["wv"], w["wo"], w["q_norm"], w["k_norm"])
    x = synth.layer_input(1, T)
    xt = torch.from_numpy(x).to(dev)
    return T, w, layer, x, xt


def wl_layer_fwd(args, dev, stream, ctx):
    import oracle

    T, w, layer, x, xt = _layer_setup(args, dev)
    d, H, D = 2048, 16, 128
    box = {}

    def step():
        box["out"] = layer.forward(xt, mode=args.mode, save_for_backward=False)

    def parity():
        ref = oracle.attention_layer_forward(x, w["wq"], w["wk"], w["wv"], w["wo"], w["q_norm"], w["k_norm"])
        return _rel(box["out"].cpu().numpy(), ref)

    def cpu(budget):
        threads, cores = _threads(16)
        med, n = _time_cpu(lambda: oracle.attention_layer_forward(x, w["wq"], w["wk"], w["wv"], w["wo"], w["q_norm"],
                                                                  w["k_norm"], nthreads=threads), budget)
        return {"value": (8 * T * d * d + algorithmic_flops(1, T, H, D)) / med / 1e12, "unit": "TFLOP/s",
                "cores": threads, "kind": "port",
                "sample": f"oracle OlmoAttention::forward fp32, x [1,{T},2048], x {n} runs (median {med * 1e3:.1f} ms), "
                f"{threads} threads of {cores} usable"}

    return dict(step=step, flops=8 * T * d * d + algorithmic_flops(1, T, H, D), tokens=T, parity=parity, cpu=cpu,
                metric=f"attention layer forward TFLOP/s + tok/s, OLMo-2-1B layer T={T}",
                data="synthetic (x ~ N(0,1) seed 2001, W ~ N(0,0.02), norms ~ 1+N(0,0.01))",
                config={"workload": f"OlmoAttention forward, x [1,{T},2048], {args.mode} core", "B": 1, "T": T,
                        "d_model": d, "H": H, "D": D})


def wl_layer_train(args, dev, stream, ctx):
    import numpy as np
    import torch

    import oracle
    from dirktensor_amd import synth

    T, w, layer, x, xt = _layer_setup(args, dev)
    d, H, D = 2048, 16, 128
    g = synth.normal(2002, x.shape)
    gt = torch.from_numpy(g).to(dev)
    box = {}

    def step():  # OlmoBlock::step order for one layer: zero_grad, forward, backward, step
        layer.zero_grad()
        layer.forward(xt, mode=args.mode)
        box["dx"] = layer.backward(gt)
        layer.step(0.0)  # lr 0 keeps the weights (and so the timed work) fixed across steps

    def parity():
        ref_dx, _ = oracle.attention_layer_backward(x, w["wq"], w["wk"], w["wv"], w["wo"], w["q_norm"], w["k_norm"], g)
        return _rel(box["dx"].cpu().numpy(), ref_dx)

    flops = 3 * 8 * T * d * d + 7 * algorithmic_flops(1, T, H, D) // 2

    def cpu(budget):
        threads, cores = _threads(16)
        med, n = _time_cpu(lambda: oracle.attention_layer_backward(x, w["wq"], w["wk"], w["wv"], w["wo"], w["q_norm"],
                                                                   w["k_norm"], g, nthreads=threads), budget)
        return {"value": flops / med / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
                "sample": f"oracle OlmoAttention forward + backward fp32, x [1,{T},2048], x {n} runs "
                f"(median {med * 1e3:.1f} ms), {threads} threads of {cores} usable"}

    return dict(step=step, flops=flops, tokens=T, parity=parity, cpu=cpu,
                metric=f"attention layer train step TFLOP/s + tok/s, OLMo-2-1B layer T={T}",
                data="synthetic (x ~ N(0,1) seed 2001, dL/dout ~ N(0,1) seed 2002, seeded weights)",
                config={"workload": f"OlmoAttention forward + backward + step, x [1,{T},2048], {args.mode}",
                        "B": 1, "T": T, "d_model": d, "H": H, "D": D})


def _model_setup(args, dev, n_layers=16, vocab=100352, hidden=8192, d=2048):
    """The end-to-end model at the OLMo-2-1B shape with weights drawn on the device
    (synth.device_model_params, seed 5100); host copies for the oracle."""
    import ctypes

    import torch

    import dirktensor_amd as dt
    from dirktensor_amd import OlmoModel, _capi, synth

    ctx = dt.default_context(0)
    h = ctypes.c_void_p()
    _capi.call("dt_model_create", ctx.handle, n_layers, d, d // 128, hidden, vocab, ctypes.byref(h))
    model = OlmoModel(ctx=ctx, _handle=h, _dims=(n_layers, d, hidden, vocab))
    host = {}
    for name, w in synth.device_model_params(dev, n_layers, vocab, hidden, d):
        torch.cuda.synchronize()
        _capi.call("dt_model_set_param", model.handle, name.encode(), w.data_ptr(), w.numel(), _capi.DT_MEM_DEVICE)
        host[name] = w.cpu().numpy()
        del w
    T = args.T if args.T != 4096 else 2048  # the end-to-end workload is quoted at T = 2048
    tok = synth.model_tokens(1, T, vocab)
    return model, host, tok, T


def _model_flops(T, n_layers=16, vocab=100352, hidden=8192, d=2048, H=16, D=128):
    gemm = n_layers * (8 * T * d * d + 6 * T * d * hidden) + 2 * T * d * vocab
    attn = n_layers * algorithmic_flops(1, T, H, D)
    return gemm, attn


def wl_model_fwd(args, dev, stream, ctx):
    import torch

    import oracle

    model, host, tok, T = _model_setup(args, dev)
    logits = torch.empty((1, T, model.vocab), dtype=torch.float32, device=dev)
    gemm, attn = _model_flops(T)
    box = {}

    def step():
        model.forward(tok, mode=args.mode, save_for_backward=False, out=logits)

    def run_oracle():  # one full forward on the host; its time is the CPU baseline's sample
        threads, _ = _threads(16)
        t0 = time.perf_counter()
        box["ref"] = oracle.model_forward(tok, host, nthreads=threads)
        box["cpu_s"] = time.perf_counter() - t0

    def parity():
        if "ref" not in box:
            run_oracle()
        return _rel(logits.cpu().numpy(), box["ref"])

    def cpu(budget):
        threads, cores = _threads(16)
        if "cpu_s" not in box:
            run_oracle()
        sec = box["cpu_s"]
        return {"value": (gemm + attn) / sec / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
                "sample": f"oracle OlmoModel::forward fp32, 16 layers, tokens [1,{T}], vocab 100352, one full run "
                f"({sec:.1f} s), {threads} threads of {cores} usable"}

    def release():  # frees the model's device memory and the host copies (the default line's extra)
        model.close()
        host.clear()
        box.clear()

    return dict(step=step, flops=gemm + attn, tokens=T, parity=parity, cpu=cpu, release=release,
                metric=f"end-to-end prefill tok/s + TFLOP/s, OLMo-2-1B (16 layers, vocab 100352) T={T}",
                data="synthetic (tokens ~ U[0,100352) seed 5001; weights drawn on the device, torch.Generator seed "
                     "5100: matrices N(0,0.02) rounded to bf16, norms 1+N(0,0.01))",
                config={"workload": f"OlmoModel forward, tokens [1,{T}], {args.mode}", "B": 1, "T": T,
                        "n_layers": 16, "d_model": 2048, "vocab": 100352, "hidden": 8192})


def wl_model_train(args, dev, stream, ctx):
    import torch

    from dirktensor_amd import ce_loss

    model, host, tok, T = _model_setup(args, dev)
    logits = torch.empty((1, T, model.vocab), dtype=torch.float32, device=dev)
    gemm, attn = _model_flops(T)
    box = {}

    def step():  # main.cpp:59-91 for one batch: forward, loss and its gradient, backward, step
        model.zero_grad()
        model.forward(tok, mode=args.mode, save_for_backward=True, out=logits)
        box["loss"], g = ce_loss(logits, tok, 100277, with_grad=True)
        model.backward(g)
        model.step(0.0)  # lr 0 keeps the weights (and so the timed work) fixed across steps

    def parity():
        import oracle

        ref = oracle.ce_loss(oracle.model_forward(tok, host, nthreads=_threads(16)[0]), tok, 100277)
        return abs(box["loss"] - ref) / abs(ref)

    return dict(step=step, flops=3 * gemm + 7 * attn // 2, tokens=T, parity=parity, cpu=lambda budget: None,
                metric=f"end-to-end train step tok/s + TFLOP/s, OLMo-2-1B (16 layers, vocab 100352) T={T}",
                data="synthetic (as the model_fwd workload)",
                config={"workload": f"OlmoModel forward + ce_loss + backward + step, tokens [1,{T}], {args.mode}",
                        "B": 1, "T": T, "n_layers": 16, "d_model": 2048, "vocab": 100352, "hidden": 8192})


WORKLOADS = {"flash_fwd": wl_flash_fwd, "flash_bwd": wl_flash_bwd, "ragged_fwd": wl_ragged_fwd,
             "layer_fwd": wl_layer_fwd, "layer_train": wl_layer_train, "model_fwd": wl_model_fwd,
             "model_train": wl_model_train}


if __name__ == "__main__":
    sys.exit(main())
