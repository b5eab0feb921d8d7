#!/usr/bin/env python3
"""Headline benchmark: fp16 x fp8-e5m2 scaled_mm on one MI355X.

One step = one launch of the scaled_mm hot path (torch.ops.feather_ops.scaled_mm,
i.e. launch_scaled_mm of libfeatherops_amd.so) on the headline shape
M=32768, K=5120, N=13824 (config 4, video-DiT FFN up-projection), fp16 out,
per-tensor scale and bias, inputs resident in HBM. The weight is a synthetic
~N(0, 0.02) fp16 matrix quantized and prepacked on the device by the
quantize kernel; A ~ N(0, 1).

Also measured in the same run (extra keys of the JSON line):
  bf16_activations  the headline shape with bf16 activations through the
              any-M op, beside fp16 activations and torch's cast + the GEMM
  small_m     config 2 (M=16, K=N=4096): GB/s, rotating over enough distinct
              weights (> 256 MB) that the Infinity Cache cannot serve them;
              torch graph replay, plus back-to-back and HIP-graph launches
              through the C ABI beside a streaming floor timed both ways;
              frac_of_floor compares the back-to-back ones (like for like)
  quantize    quantize+prepack of a 13824x5120 fp16 weight (config 5's op, the
              one-pass kernel), four weights in rotation so they stream from
              HBM; GB/s on the 3 B per element minimum
  hbm_aux     the bf16 -> fp16 casts (N x N, N = 1024 .. 16384) and the
              dequantize of a 13824x5120 weight, as GB/s
  reference_published_shape  8192^3 on the reference's published config
              tuple and on the 256x256 tile (context only)
  lora        an unmerged rank-64 LoRA layer on the headline shape, fused
              epilogue against the reference's separate pass
  configs     every benchmark workload at one GPU: C1 (M=256, K=N=1024), C3
              (image-DiT linears, M=4096, bf16 out), C4 (video-DiT linears,
              M=32768), C5 (40-block x 6-linear stack at M=32768: on-device
              quantize+prepack of all 240 weights, then the 240 GEMMs); each
              GEMM shape on the best of a few gfx950 tile configs (what the
              autotuner picks), as TFLOP/s and fraction of the fp16 MFMA peak
  cpu_baseline  the oracle's host-torch restatement of kernel/naive.py (fp16
              CPU matmul) on up to 16 host cores, on a bounded sample of the
              headline rows

The headline is W untimed warmup steps, then K timed steps between HIP events.
Every extra key runs ~25 ms untimed before ~25 ms of timed calls
(time_steady): its kernels are short against the tens of ms the engine clock
takes to rise under load.

Usage: python bench.py [--gpus 1] [--steps 20] [--warmup 5] [--no-cpu]
"""

from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time
from pathlib import Path

REPO = Path(__file__).resolve().parent
sys.path.insert(0, str(REPO))

PEAK_FP16_TFLOPS = 2500.0  # MI355X dense fp16 MFMA
PEAK_HBM_GBPS = 8000.0  # MI355X HBM3E
METRIC = "TFLOPS & % fp16-MFMA peak, fp16×e5m2 GEMM M32768 K5120 N13824; GB/s at M=16"
HEADLINE_CFG = (2, 4, 4, 8, 4)
TRAFFIC_FILE = REPO / "profiles" / "scaled_mm_lds256_headline_pmc.txt"


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def gemm_bytes(M: int, N: int, K: int) -> int:
    """Algorithmic bytes of one call (reference cpp bench formula): A fp16 + B fp8 + C fp16."""
    return 2 * M * K + N * K + 2 * M * N


def _quantized_weight(N, K, seed, dev, quant):
    import torch

    g = torch.Generator(device=dev).manual_seed(seed)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.02).half()
    qt = quant.make_feather_quantized_weight(w, None, torch.float16)
    return quant.get_feather_plain_tensors(qt)


def time_launches(fn, n: int):
    """Average ms per call of n back-to-back calls, bracketed by HIP events on the current stream."""
    import torch

    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    s.record()
    for i in range(n):
        fn(i)
    e.record()
    torch.cuda.synchronize()
    return s.elapsed_time(e) / n


def time_steady(fn, min_calls: int = 3, window_ms: float = 25.0):
    """Average ms per call at a warmed-up engine clock: fn runs untimed for about window_ms, then
    at least min_calls calls covering about window_ms are timed with time_launches. (The clock
    rises over the first tens of ms under load; a short timed region right after a
    synchronisation measures that ramp: a 60 us GEMM timed over 10 calls reads ~15% slow.)"""
    import math

    one = time_launches(fn, 1)
    n = max(min_calls, math.ceil(window_ms / max(one, 1e-3)))
    for i in range(n):
        fn(i)
    return time_launches(fn, n)


def streaming_floor_us(nbytes: int, graph: bool = False):
    """Per-call time of a plain read-only streaming kernel over nbytes (24 rotated buffers),
    measured by the C++ bench in a child process (back-to-back launches, or with graph=True
    the 24 launches replayed from a HIP graph); None if it is not built."""
    import subprocess

    exe = REPO / "comfyui-featherops_amd" / "cpp_benchmarks" / "build" / "benchmark_hbm_copy"
    if not exe.exists():
        return None
    try:
        out = subprocess.run([str(exe), "--read-bytes", str(nbytes)] + (["--graph"] if graph else []),
                             capture_output=True, text=True, timeout=120)
    except (OSError, subprocess.TimeoutExpired):
        return None
    m = re.search(r"([0-9.]+) us/call", out.stdout)
    return float(m.group(1)) if out.returncode == 0 and m else None


def cpp_bench_us(M: int, N: int, K: int, rotate: int = 24, iters: int = 5000):
    """Per-call times of the small-M GEMM through the C ABI (cpp_benchmarks/benchmark_scaled_mm_hip,
    rotate distinct weights, fp16 out, scale and bias): (back-to-back launches, the rotate launches
    replayed from a HIP graph) -- the two launch methods streaming_floor_us offers; None if the
    bench is not built."""
    import subprocess

    exe = REPO / "comfyui-featherops_amd" / "cpp_benchmarks" / "build" / "benchmark_scaled_mm_hip"
    if not exe.exists():
        return None
    cmd = [str(exe), "--m", str(M), "--n", str(N), "--k", str(K), "--rotate", str(rotate), "--warmup",
           str(iters // 4), "--iters", str(iters)]
    try:
        out = subprocess.run(cmd, capture_output=True, text=True, timeout=120)
    except (OSError, subprocess.TimeoutExpired):
        return None
    m = re.search(r"back-to-back us: ([0-9.]+)", out.stdout)
    mg = re.search(r"graph-replay us: ([0-9.]+)", out.stdout)
    if out.returncode != 0 or not m or not mg:
        return None
    return float(m.group(1)), float(mg.group(1))


def _cpp_bench(args, key: str, timeout: int = 180):
    """Run the C++ bench with args in a child process and return the float after `key`."""
    import subprocess

    exe = REPO / "comfyui-featherops_amd" / "cpp_benchmarks" / "build" / "benchmark_scaled_mm_hip"
    if not exe.exists():
        return None
    try:
        out = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=timeout)
    except (OSError, subprocess.TimeoutExpired):
        return None
    m = re.search(re.escape(key) + r"\s*([0-9.]+)", out.stdout)
    return float(m.group(1)) if out.returncode == 0 and m else None


def bench_hbm_aux() -> dict:
    """The HBM-bound auxiliary kernels, each timed as back-to-back launches over rotated
    buffers (at least ~1 GB in total, so the 256 MB Infinity Cache does not serve them):
    bf16 -> fp16 (round toward zero, reference kernel/convert.py, and round to nearest even,
    the any-M entry's cast) on N x N for the N of the reference's benchmark_convert.py:39-53,
    GB/s on its 4 B per element; dequantize of the headline 13824 x 5120 weight to fp16
    (3 B per element)."""
    import math

    out = {"timing": "C++ bench (cpp_benchmarks/benchmark_scaled_mm_hip --convert / --dequant), back-to-back "
                     "launches between two HIP events, inputs and outputs rotated over >= 1 GB"}
    for mode in ("rtz", "rne"):
        rows = {}
        for n in (1024, 2048, 4096, 8192, 16384):
            nbytes = 4 * n * n
            rot = min(256, max(2, math.ceil(1.0e9 / nbytes)))
            iters = max(50, int(0.02 * 5e12 / nbytes))
            us = _cpp_bench(["--convert", mode, "--n", n, "--rotate", rot, "--warmup", iters // 4 + rot, "--iters",
                             iters], "back-to-back us:")
            if us is None:
                continue
            gbps = nbytes / (us * 1e-6) / 1e9
            rows[str(n)] = {"us": round(us, 3), "GB_per_s": round(gbps, 1),
                            "frac_hbm_peak": round(gbps / PEAK_HBM_GBPS, 4), "rotated": rot}
        out["bf16_to_fp16_" + mode] = rows
    Nd, Kd = 13824, 5120
    us = _cpp_bench(["--dequant", "--n", Nd, "--k", Kd, "--rotate", 5, "--warmup", 20, "--iters", 200],
                    "back-to-back us:")
    if us is not None:
        gbps = 3 * Nd * Kd / (us * 1e-6) / 1e9
        out["dequantize_e5m2"] = {"N": Nd, "K": Kd, "out": "float16", "us": round(us, 2), "GB_per_s": round(gbps, 1),
                                  "frac_hbm_peak": round(gbps / PEAK_HBM_GBPS, 4), "rotated": 5,
                                  "bytes_model": "1 B read + 2 B written per element"}
    return out


def bench_reference_published_shape() -> dict:
    """The reference's one published figure for this path (docs/benchmark_tracking.md:12-21:
    M = N = K = 8192, config (1,8,4,8,2), scale and bias, fp16 out, 45.5-45.9 TFLOP/s on a
    gfx1151 iGPU) on this GPU: the same config tuple and the 256x256 gfx950 tile, through the C++ bench
    (the reference's own bench recipe). Different hardware: context, not a target."""
    out = {"shape": "M=N=K=8192, fp16 out, scale+bias", "reference_published_TFLOP_per_s": [45.5, 45.9],
           "reference_hardware": "gfx1151 (Strix Halo iGPU), docs/benchmark_tracking.md:12-21",
           "note": "different hardware: context only, not a target"}
    for name, cfg in (("config_1_8_4_8_2", (1, 8, 4, 8, 2)), ("config_2_4_4_8_4_gfx950_256x256", (2, 4, 4, 8, 4))):
        tf = _cpp_bench(["--m", 8192, "--n", 8192, "--k", 8192, "--warps_m", cfg[0], "--warps_n", cfg[1],
                         "--unroll", cfg[2], "--repeat_m", cfg[3], "--repeat_n", cfg[4], "--warmup", 20,
                         "--iters", 100], "back-to-back ms:")
        if tf is not None:
            ms = tf
            out[name] = {"ms": round(ms, 4), "TFLOP_per_s": round(2 * 8192 ** 3 / (ms * 1e-3) / 1e12, 1)}
    return out


def read_traffic():
    """HBM bytes per headline launch from the committed rocprofv3 PMC summary, if present."""
    if not TRAFFIC_FILE.exists():
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*([0-9.eE+]+)", TRAFFIC_FILE.read_text(), flags=re.M)
    return float(m.group(1)) if m else None


def _cpu_model() -> str:
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(budget_s: float = 12.0):
    """The host-torch restatement of kernel/naive.py (unpack, e5m2 -> fp16, fp16 CPU matmul,
    scale in fp32, cast, bias) on the host cores, over a growing number of headline rows until
    ~budget_s of work is timed. Threads: the host's cores, at most 16 (a one-GPU box's share)."""
    import numpy as np
    import torch

    from oracle import feather_oracle as O

    threads = max(1, min(os.cpu_count() or 1, 16))
    prev_threads = torch.get_num_threads()
    torch.set_num_threads(threads)
    M, N, K = 32768, 13824, 5120
    g = torch.Generator().manual_seed(0)
    w = torch.randn(N, K, generator=g) * 0.02
    s = np.float32(w.abs().max().item()) / np.float32(57344.0)
    codes = (w * float(np.float32(1.0) / s)).to(torch.float8_e5m2).view(torch.uint8)
    packed = codes.view(N, K // 16, 16).permute(1, 0, 2).contiguous()
    bias = (torch.randn(N, generator=g) * 0.01).half()
    st = torch.tensor(s)
    O.scaled_mm_naive_torch(torch.randn(16, K, generator=g).half(), packed, st, bias, torch.float16)  # warm
    rows = 64
    total_t, total_rows = 0.0, 0
    try:
        while True:
            a = torch.randn(rows, K, generator=g).half()
            t0 = time.perf_counter()
            O.scaled_mm_naive_torch(a, packed, st, bias, torch.float16)
            dt = time.perf_counter() - t0
            total_t, total_rows = total_t + dt, total_rows + rows
            if total_t >= budget_s or rows >= 4096:
                break
            rows *= 2
    finally:
        torch.set_num_threads(prev_threads)
    tflops = 2.0 * total_rows * N * K / total_t / 1e12
    # beside it: the same steps with the product taken by the fp32 BLAS matmul and rounded to
    # fp16 (the oracle's numpy formulation of naive.py), which does not depend on whether the host
    # CPU has a native fp16 matmul path; the weight is decoded once, outside the timed region
    torch.set_num_threads(threads)
    w32 = packed.transpose(1, 2).reshape(K, N).view(torch.float8_e5m2).float()
    t_blas, blas_rows, rows = 0.0, 0, 256
    try:
        while t_blas < budget_s / 2 and blas_rows < 8192:
            a = torch.randn(rows, K, generator=g).half()
            t0 = time.perf_counter()
            y = ((a.float() @ w32).half().float() * st).half() + bias
            t_blas += time.perf_counter() - t0
            blas_rows += rows
            rows *= 2
    finally:
        torch.set_num_threads(prev_threads)
    del w32, y
    blas_tflops = 2.0 * blas_rows * N * K / t_blas / 1e12
    return {"value": round(tflops, 4), "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "cpu_model": _cpu_model(), "os_cpu_count": os.cpu_count(), "torch_threads": threads,
            "sample": f"host-torch restatement of kernel/naive.py (fp16 CPU matmul, torch {torch.__version__}) "
                      f"on {total_rows} of the {M} headline rows, K={K}, N={N}, {total_t:.1f} s",
            "full_job_seconds_extrapolated": round(total_t * M / total_rows, 1),
            "fp32_blas_variant": {"value": round(blas_tflops, 4), "unit": "TFLOP/s", "rows": blas_rows,
                                  "seconds": round(t_blas, 1),
                                  "what": "naive.py's steps with the product from the fp32 BLAS matmul rounded "
                                          "to fp16 (the oracle's numpy formulation); weight decoded once, untimed"}}


CANDIDATE_CFGS = [(2, 4, 4, 8, 4), (4, 2, 4, 4, 8), (2, 4, 4, 8, 3), (2, 4, 4, 4, 6), (2, 2, 4, 4, 4)]


def _gemm_shape(dev, op, quant, g, M, N, K, out_dtype, seed, reps=10):
    """Best time over the candidate tile configs for one shape (scale and bias on)."""
    import torch

    bp, scale = _quantized_weight(N, K, seed, dev, quant)
    a = torch.randn(M, K, generator=g, device=dev).half()
    bias = (torch.randn(N, generator=g, device=dev) * 0.01).to(out_dtype)
    c = torch.empty(M, N, dtype=out_dtype, device=dev)
    best = None
    for cfg in CANDIDATE_CFGS:
        wm, wn, u, rm, rn = cfg
        if M % (16 * wm * rm) or N % (16 * wn * rn) or K % (16 * u):
            continue  # the op keeps the reference's block-divisibility rule
        fn = lambda _i, cfg=cfg: op(a, bp, scale, bias, c, *cfg, 1)  # noqa: E731
        ms = time_steady(fn, reps)
        if best is None or ms < best[0]:
            best = (ms, cfg)
    ms, cfg = best
    tflops = 2.0 * M * N * K / (ms * 1e-3) / 1e12
    return {"M": M, "N": N, "K": K, "out": str(out_dtype).replace("torch.", ""), "ms": round(ms, 4),
            "TFLOP_per_s": round(tflops, 1), "frac_fp16_peak": round(tflops / PEAK_FP16_TFLOPS, 4),
            "config": list(cfg)}, cfg


def bench_configs(dev, op, quant, g):
    """Every benchmark workload on this GPU (see the module docstring)."""
    import torch

    out = {}
    # C1: the CPU-reference case on the GPU (tiny: launch-bound, timed by HIP graph replay)
    M1, N1, K1 = 256, 1024, 1024
    bp, scale = _quantized_weight(N1, K1, 7, dev, quant)
    a1 = torch.randn(M1, K1, generator=g, device=dev).half()
    c1 = torch.empty(M1, N1, dtype=torch.float16, device=dev)
    best = None
    for cfg in [(2, 2, 4, 4, 4), (1, 4, 4, 4, 2), (2, 4, 4, 4, 4)]:
        op(a1, bp, scale, None, c1, *cfg, 1)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                op(a1, bp, scale, None, c1, *cfg, 1)
        graph.replay()
        ms = time_steady(lambda _i: graph.replay(), 10) / 20
        if best is None or ms < best[0]:
            best = (ms, cfg)
    tf = 2.0 * M1 * N1 * K1 / (best[0] * 1e-3) / 1e12
    out["c1"] = {"M": M1, "N": N1, "K": K1, "out": "float16", "us": round(best[0] * 1e3, 2), "TFLOP_per_s": round(tf, 2),
                 "frac_fp16_peak": round(tf / PEAK_FP16_TFLOPS, 5), "config": list(best[1]),
                 "timing": "HIP graph replay (launch-bound size)"}
    log(f"bench: C1 {best[0] * 1e3:.2f} us, {tf:.1f} TFLOP/s")

    # C3: image-DiT linears, M=4096, bf16 out
    c3 = {}
    for name, (K, N) in {"qkvo_3072x3072": (3072, 3072), "up_3072x12288": (3072, 12288),
                         "down_12288x3072": (12288, 3072)}.items():
        c3[name], _ = _gemm_shape(dev, op, quant, g, 4096, N, K, torch.bfloat16, 11)
    set_ms = 4 * c3["qkvo_3072x3072"]["ms"] + c3["up_3072x12288"]["ms"] + c3["down_12288x3072"]["ms"]
    set_flop = 2.0 * 4096 * (4 * 3072 * 3072 + 2 * 3072 * 12288)
    c3["set"] = {"linears": "4 x (3072->3072) + (3072->12288) + (12288->3072)", "ms": round(set_ms, 4),
                 "TFLOP_per_s": round(set_flop / (set_ms * 1e-3) / 1e12, 1)}
    out["c3"] = c3
    log(f"bench: C3 set {set_ms:.3f} ms, {c3['set']['TFLOP_per_s']} TFLOP/s")

    # C4: video-DiT-14B linears, M=32768, fp16 out
    c4 = {}
    cfg4 = {}
    for name, (K, N) in {"qkvo_5120x5120": (5120, 5120), "up_5120x13824": (5120, 13824),
                         "down_13824x5120": (13824, 5120)}.items():
        c4[name], cfg4[(K, N)] = _gemm_shape(dev, op, quant, g, 32768, N, K, torch.float16, 13, reps=5)
    set_ms = 4 * c4["qkvo_5120x5120"]["ms"] + c4["up_5120x13824"]["ms"] + c4["down_13824x5120"]["ms"]
    set_flop = 2.0 * 32768 * (4 * 5120 * 5120 + 2 * 5120 * 13824)
    c4["set"] = {"linears": "4 x (5120->5120) + (5120->13824) + (13824->5120)", "ms": round(set_ms, 4),
                 "TFLOP_per_s": round(set_flop / (set_ms * 1e-3) / 1e12, 1)}
    out["c4"] = c4
    log(f"bench: C4 set {set_ms:.3f} ms, {c4['set']['TFLOP_per_s']} TFLOP/s")

    # C5: 40 blocks x {q, k, v, o, ffn_up, ffn_down}; every weight generated,
    # then quantized+prepacked on the device (timed), then the 240 GEMMs in
    # block order (timed as one region). Each linear reads a fixed ~N(0,1)
    # input of its K (no un-normalised chaining of random layers).
    M5, H, F = 32768, 5120, 13824
    layer_shapes = [(H, H)] * 4 + [(H, F), (F, H)]  # (K, N)
    xs = {H: torch.randn(M5, H, generator=g, device=dev).half(), F: torch.randn(M5, F, generator=g, device=dev).half()}
    outs = {H: torch.empty(M5, H, dtype=torch.float16, device=dev), F: torch.empty(M5, F, dtype=torch.float16, device=dev)}
    # all 240 fp16 weights are generated first, then quantized back to back
    # between two events (one region, so host-side dispatch overlaps the
    # device work instead of being timed per weight)
    raw = []
    for blk in range(40):
        for li, (K, N) in enumerate(layer_shapes):
            gw = torch.Generator(device=dev).manual_seed(1000 + 6 * blk + li)
            w = (torch.randn(N, K, generator=gw, device=dev) * 0.02).half()
            b5 = (torch.randn(N, generator=gw, device=dev) * 0.01).half()
            raw.append((K, N, w, b5))
    # one untimed pass first, so that the timed one takes its output buffers
    # from torch's caching allocator instead of timing fresh device allocations
    qts = [quant.make_feather_quantized_weight(w, None, torch.float16) for _, _, w, _ in raw]
    del qts
    torch.cuda.synchronize()
    # three eager passes: torch's caching allocator now and then frees and
    # re-maps device memory inside such a pass (a pass then takes ~4x longer
    # with the host blocked in the allocator); the best pass is reported with
    # all three
    q_passes = []
    for rep in range(3):
        if rep:
            del qts
            torch.cuda.synchronize()
        ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        ev0.record()
        qts = [quant.make_feather_quantized_weight(w, None, torch.float16) for _, _, w, _ in raw]
        ev1.record()
        ev1.synchronize()
        q_passes.append(ev0.elapsed_time(ev1))
    q_ms = min(q_passes)
    # the same 240 calls captured in a HIP graph and replayed: the device time
    # alone (no launch gaps, no allocator)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        qts_graph = [quant.make_feather_quantized_weight(w, None, torch.float16) for _, _, w, _ in raw]
    graph.replay()
    torch.cuda.synchronize()
    q_dev_ms = time_launches(lambda _i: graph.replay(), 3)
    del graph, qts_graph
    weights = []
    for (K, N, w, b5), qt in zip(raw, qts):
        bp5, s5 = quant.get_feather_plain_tensors(qt)
        weights.append((K, N, bp5, s5, b5))
    del raw, qts
    torch.cuda.synchronize()

    def run_stack(_i):
        for K, N, bp5, s5, b5 in weights:
            op(xs[K], bp5, s5, b5, outs[N], *cfg4[(K, N)], 1)

    run_stack(0)
    gemm_ms = time_launches(run_stack, 1)
    flop5 = 40 * 2.0 * M5 * (4 * H * H + 2 * H * F)
    elems = 40 * (4 * H * H + 2 * H * F)
    out["c5"] = {"blocks": 40, "linears": 240, "M": M5, "quantize_ms_total": round(q_ms, 2),
                 "quantize_GB_per_s": round(elems * 3 / (q_ms * 1e-3) / 1e9, 1),
                 "quantize_device_ms_total": round(q_dev_ms, 2),
                 "quantize_device_GB_per_s": round(elems * 3 / (q_dev_ms * 1e-3) / 1e9, 1),
                 "quantize_bytes_model": "3 B per element (2 B read + 1 B written)",
                 "quantize_eager_passes_ms": [round(x, 2) for x in q_passes],
                 "quantize_timing": "eager: 240 calls between two events (host dispatch included), best of three "
                                    "passes; device: the same calls replayed from a HIP graph",
                 "gemm_ms_total": round(gemm_ms, 2), "gemm_TFLOP_per_s": round(flop5 / (gemm_ms * 1e-3) / 1e12, 1),
                 "gemm_frac_fp16_peak": round(flop5 / (gemm_ms * 1e-3) / 1e12 / PEAK_FP16_TFLOPS, 4),
                 "end_to_end_ms": round(q_ms + gemm_ms, 2),
                 "weights_GB_e5m2": round(elems / 1e9, 2)}
    log(f"bench: C5 quantize {q_ms:.1f} ms eager, {q_dev_ms:.1f} ms device, GEMMs {gemm_ms:.1f} ms "
        f"({out['c5']['gemm_TFLOP_per_s']} TFLOP/s)")
    del weights, xs, outs
    torch.cuda.empty_cache()
    return out


def bench_lora(dev, hk, g) -> dict:
    """Unmerged LoRA (comfy_feather/lora.py) on the headline shape, bf16
    activations and output, one rank-64 basic patch: the whole layer with the
    term fused into the GEMM epilogue (T build + fused GEMM) against the
    reference's separate pass (GEMM, then y += F.linear(F.linear(x, A), B) * s)."""
    import importlib
    from types import SimpleNamespace

    import torch

    lora = importlib.import_module("featherops_amd.comfy_feather.lora")
    M, N, K, R = 32768, 13824, 5120, 64
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    bp = hk.prepack_b_for_scaled_mm((torch.randn(K, N, generator=g, device=dev) * 0.02).to(torch.float8_e5m2))
    s = torch.tensor(1.0, device=dev)
    bias = torch.zeros(N, dtype=torch.bfloat16, device=dev)
    down = (torch.randn(R, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    up = (torch.randn(N, R, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    wf = [SimpleNamespace(patches={"w": [(1.0, SimpleNamespace(weights=(up, down, float(R), None)), 1.0)]}, key="w")]

    def fused(_i):
        t, u, x16 = lora.lora_layer_inputs(x, wf)  # what Linear.forward runs
        return hk.scaled_mm_hip_any_m_lora(x16, bp, s, bias, torch.bfloat16, t, u)

    def separate(_i):
        y = hk.scaled_mm_hip_any_m(x, bp, s, bias, torch.bfloat16)
        return lora.apply_lora_patches(x, y, wf)

    ms_f = time_steady(fused, 5)
    ms_s = time_steady(separate, 5)
    log(f"bench: LoRA rank {R} layer fused {ms_f:.3f} ms, separate {ms_s:.3f} ms")
    return {"M": M, "N": N, "K": K, "rank": R, "dtype": "bf16", "fused_layer_ms": round(ms_f, 4),
            "separate_layer_ms": round(ms_s, 4), "speedup": round(ms_s / ms_f, 3)}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--only-headline", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only: --gpus {args.gpus} is not supported on this single-GPU build "
              "(the kernel runs on one GPU's shard; multi-GPU sharding is design-only here)", file=sys.stderr)
        return 2

    import numpy as np
    import torch

    import __graft_entry__

    __graft_entry__.load_package()
    import importlib

    hk = importlib.import_module("featherops_amd.kernel.hip.hip_kernel")
    quant = importlib.import_module("featherops_amd.comfy_feather.quant")
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)

    # ---------------- headline GEMM ----------------
    M, N, K = 32768, 13824, 5120
    log(f"bench: headline M={M} N={N} K={K} cfg={HEADLINE_CFG}")
    bp, scale = _quantized_weight(N, K, 1, dev, quant)
    g = torch.Generator(device=dev).manual_seed(2)
    a = torch.randn(M, K, generator=g, device=dev).half()
    bias = (torch.randn(N, generator=g, device=dev) * 0.01).half()
    c = torch.empty(M, N, dtype=torch.float16, device=dev)
    op = torch.ops.feather_ops.scaled_mm.default

    def step(_i):
        op(a, bp, scale, bias, c, *HEADLINE_CFG, 1)

    for i in range(args.warmup):
        step(i)
    torch.cuda.synchronize()
    ms = time_launches(step, args.steps)
    flops = 2.0 * M * N * K
    tflops = flops / (ms * 1e-3) / 1e12
    assert torch.isfinite(c).all().item(), "non-finite output in the headline GEMM"
    log(f"bench: headline {ms:.3f} ms/step, {tflops:.1f} TFLOP/s ({100 * tflops / PEAK_FP16_TFLOPS:.1f}% of peak)")
    traffic = read_traffic()
    result = {
        "metric": METRIC,
        "value": round(tflops, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp16",
        "data": "synthetic (A ~ N(0,1) fp16; W ~ N(0,0.02) fp16 quantized+prepacked on device to e5m2)",
        "config": {"workload": "scaled_mm fp16 x e5m2, M32768 K5120 N13824, fp16 out, scale+bias "
                               "(the C4 video-DiT up-projection, the headline)",
                   "M": M, "N": N, "K": K, "out_dtype": "fp16", "kernel_config": list(HEADLINE_CFG)},
        "pct_fp16_mfma_peak": round(100 * tflops / PEAK_FP16_TFLOPS, 2),
        "roofline": {"bound": "mfma", "achieved": round(tflops, 2), "peak": PEAK_FP16_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(tflops / PEAK_FP16_TFLOPS, 4), "traffic": traffic,
                     "algorithmic_bytes": gemm_bytes(M, N, K)},
    }
    if not args.only_headline:
        # context: the vendor fp16 x fp16 GEMM (torch.matmul -> hipBLASLt) on the same shape
        b16 = torch.randn(K, N, generator=g, device=dev).half()
        for _ in range(2):
            torch.matmul(a, b16)
        ms_ref = time_launches(lambda _i: torch.matmul(a, b16), max(3, args.steps // 2))
        result["context_fp16xfp16_torch_matmul"] = {"ms": round(ms_ref, 4),
                                                    "TFLOP_per_s": round(flops / (ms_ref * 1e-3) / 1e12, 2)}
        log(f"bench: torch fp16 matmul (hipBLASLt) same shape {ms_ref:.3f} ms")
        del b16

        # bf16 activations on the headline shape through the any-M op (the
        # large tiles round them to fp16 with the library's RNE cast pass, then
        # run the fp16 GEMM), beside the reference's route: x.to(float16)
        # (comfy_feather/ops.py:88) followed by the same GEMM
        abf = a.to(torch.bfloat16)
        any_m = torch.ops.feather_ops.scaled_mm_any_m.default
        for _ in range(2):
            any_m(abf, bp, scale, bias, torch.float16)
        # the three routes alternate over three passes (each the best of its passes), so that a drift
        # of the engine clock over the run does not favour whichever is timed first
        n_bf = max(3, args.steps // 2)
        routes = {"bf16": lambda _i: any_m(abf, bp, scale, bias, torch.float16),
                  "fp16": lambda _i: any_m(a, bp, scale, bias, torch.float16),
                  "torch_cast": lambda _i: any_m(abf.to(torch.float16), bp, scale, bias, torch.float16)}
        best_ms = {k: float("inf") for k in routes}
        for _ in range(3):
            for k, fn in routes.items():
                best_ms[k] = min(best_ms[k], time_launches(fn, n_bf))
        ms_bf, ms_f16, ms_refroute = best_ms["bf16"], best_ms["fp16"], best_ms["torch_cast"]
        result["bf16_activations"] = {"ms": round(ms_bf, 4), "fp16_activations_ms": round(ms_f16, 4),
                                      "torch_cast_then_gemm_ms": round(ms_refroute, 4),
                                      "overhead_vs_fp16": round(ms_bf / ms_f16 - 1.0, 4),
                                      "timing": f"best of three alternating passes of {n_bf} calls each",
                                      "route": "library RNE cast pass + fp16 GEMM (any-M op)"}
        log(f"bench: bf16 activations {ms_bf:.3f} ms (fp16 {ms_f16:.3f}, torch cast + GEMM {ms_refroute:.3f})")
        del abf
    del a, c

    if not args.only_headline:
        # ---------------- small M (config 2), weight rotation past the 256 MB MALL ----------------
        Ms, Ns, Ks = 16, 4096, 4096
        nrot = 24  # 24 x 16.8 MB = 403 MB of distinct weights
        log(f"bench: small-M M={Ms} N={Ns} K={Ks}, rotating {nrot} weights")
        ws = [_quantized_weight(Ns, Ks, 100 + r, dev, quant) for r in range(nrot)]
        a16 = torch.randn(Ms, Ks, generator=g, device=dev).half()
        b16 = (torch.randn(Ns, generator=g, device=dev) * 0.01).half()
        c16 = torch.empty(Ms, Ns, dtype=torch.float16, device=dev)

        def step16(i):
            w, s = ws[i % nrot]
            op(a16, w, s, b16, c16, 1, 1, 2, 1, 2, 1)

        for i in range(2 * nrot):
            step16(i)
        torch.cuda.synchronize()
        # a ~3-5 us kernel is shorter than one Python dispatch, so the calls are
        # captured once in a HIP graph (ten rounds over the rotated weights: 240
        # launches, so the per-replay cost of torch's graph launch is spread over
        # many calls) and the graph is replayed: the timed region then holds device
        # work only
        rounds = 10
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for i in range(nrot * rounds):
                step16(i)
        graph.replay()
        torch.cuda.synchronize()
        ms16 = time_steady(lambda _i: graph.replay(), 4) / (nrot * rounds)
        eager_ms16 = time_launches(step16, 4 * nrot)
        gbps = gemm_bytes(Ms, Ns, Ks) / (ms16 * 1e-3) / 1e9
        log(f"bench: small-M {ms16 * 1e3:.2f} us/call (graph replay), {gbps:.0f} GB/s; eager {eager_ms16 * 1e3:.2f} us")
        result["small_m"] = {"M": Ms, "N": Ns, "K": Ks, "us_per_call": round(ms16 * 1e3, 3),
                             "GB_per_s": round(gbps, 1), "pct_hbm_peak": round(100 * gbps / PEAK_HBM_GBPS, 2),
                             "weights_rotated": nrot,
                             "timing": "torch CUDAGraph of 240 calls (10 rounds over the rotated weights) replayed, "
                                       "~25 ms warm-up then ~25 ms timed",
                             "eager_us_per_call": round(eager_ms16 * 1e3, 3)}
        del ws
        floor = streaming_floor_us(gemm_bytes(Ms, Ns, Ks))
        if floor is not None:
            result["small_m"]["floor_us"] = round(floor, 3)
            # the floor is timed back to back; against torch's graph replay (a different launch method)
            result["small_m"]["frac_of_floor_torch_graph"] = round(floor / (ms16 * 1e3), 3)
            result["small_m"]["frac_of_floor"] = result["small_m"]["frac_of_floor_torch_graph"]
            result["small_m"]["frac_of_floor_method"] = "floor back to back / torch graph replay of the op"
            result["small_m"]["floor"] = ("read-only streaming kernel over the same byte count, 24 rotated buffers, "
                                          "back to back (cpp_benchmarks/benchmark_hbm_copy --read-bytes)")
            log(f"bench: streaming floor for {gemm_bytes(Ms, Ns, Ks)} B: {floor:.2f} us/call")
        floor_g = streaming_floor_us(gemm_bytes(Ms, Ns, Ks), graph=True)
        if floor_g is not None:
            # the same floor with its 24 launches replayed from a HIP graph
            result["small_m"]["floor_graph_us"] = round(floor_g, 3)
            log(f"bench: streaming floor, graph replay: {floor_g:.2f} us/call")
        cpp = cpp_bench_us(Ms, Ns, Ks, nrot)
        if cpp is not None:
            # the floor's two launch methods applied to the GEMM through the C ABI: the like-for-like
            # ratios (torch's graph replay above adds ~0.5 us per node over a plain HIP graph)
            b2b, gr = cpp
            result["small_m"]["back_to_back_us_per_call"] = round(b2b, 3)
            result["small_m"]["hip_graph_us_per_call"] = round(gr, 3)
            if floor is not None:
                result["small_m"]["frac_of_floor_back_to_back"] = round(floor / b2b, 3)
                # like for like: the floor and the GEMM launched the same way
                result["small_m"]["frac_of_floor"] = result["small_m"]["frac_of_floor_back_to_back"]
                result["small_m"]["frac_of_floor_method"] = "both back to back through the C ABI (like for like)"
            if floor_g is not None:
                result["small_m"]["frac_of_floor_hip_graph"] = round(floor_g / gr, 3)
            log(f"bench: small-M through the C ABI: back to back {b2b:.2f} us/call, HIP graph {gr:.2f} us/call")

        # ---------------- quantize + prepack (config 5's on-device op) ----------------
        # four distinct 141.6 MB weights (566 MB) in rotation, so the weight is streamed from HBM
        # rather than served by the 256 MB Infinity Cache; the cache-resident rate beside it
        Nq, Kq = 13824, 5120
        nq = 4
        wqs = [(torch.randn(Nq, Kq, generator=g, device=dev) * 0.02).half() for _ in range(nq)]

        def stepq(i):
            quant.make_feather_quantized_weight(wqs[i % nq], None, torch.float16)

        for i in range(nq):
            stepq(i)
        msq = time_steady(stepq, 4 * nq)
        qbytes = Nq * Kq * (2 + 1)  # the weight read once, the e5m2 codes written once
        cus = torch.cuda.get_device_properties(dev).multi_processor_count
        share = -(-((Kq // 16 + 15) // 16) * ((Nq + 63) // 64) // cus)  # 64 x 256 blocks per workgroup
        hbm_per_elem = 3 + 2 * max(share - 12, 0) / share  # blocks beyond the 12 held (registers, LDS) read twice
        result["quantize"] = {"N": Nq, "K": Kq, "ms_per_weight": round(msq, 4),
                              "GB_per_s": round(qbytes / (msq * 1e-3) / 1e9, 1),
                              "pct_hbm_peak": round(100 * qbytes / (msq * 1e-3) / 1e9 / PEAK_HBM_GBPS, 2),
                              "GB_per_s_two_pass_bytes": round(Nq * Kq * 5 / (msq * 1e-3) / 1e9, 1),
                              "weights_rotated": nq, "timing": "eager calls between two events (~25 ms warm-up, then "
                                                               "~25 ms timed), weights rotated through 566 MB "
                                                               "(streamed from HBM)",
                              "bytes_model": "3 B per element: 2 B read + 1 B written (the minimum); "
                                             "GB_per_s_two_pass_bytes counts the two-pass path's 5 B",
                              "hbm_bytes_per_element_model": round(hbm_per_elem, 2)}
        log(f"bench: quantize {msq:.3f} ms per 13824x5120 weight (rotated)")
        del wqs

    if not args.only_headline:
        log("bench: HBM auxiliary kernels (convert, dequantize) ...")
        result["hbm_aux"] = bench_hbm_aux()
        for mode in ("rtz", "rne"):
            r = result["hbm_aux"].get("bf16_to_fp16_" + mode, {}).get("16384")
            if r:
                log(f"bench: bf16->fp16 {mode} 16384^2 {r['us']:.1f} us, {r['GB_per_s']:.0f} GB/s")
        log("bench: reference published shape 8192^3 ...")
        result["reference_published_shape"] = bench_reference_published_shape()
        result["lora"] = bench_lora(dev, hk, g)
        result["configs"] = bench_configs(dev, op, quant, g)

    if not args.no_cpu:
        log("bench: CPU baseline (host-torch naive restatement) ...")
        result["cpu_baseline"] = cpu_baseline()
    else:
        result["cpu_baseline"] = None

    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
