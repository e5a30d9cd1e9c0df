#!/usr/bin/env python3
"""Benchmark of the w8g64 quantized linear on one MI355X.

Headline (BASELINE.json metric): the video feed-forward pair of config 2 --
X [8160 x 4096] bf16 -> up 4096->16384 w8g64 with GELU-tanh fused -> down
16384->4096 w8g64 -- reported as TFLOP/s over both GEMMs and as a fraction
of the bf16 dense MFMA peak. A "step" is one pass of that pair over one
batch of synthetic input already resident in HBM.

Also reported on the same line:
  audio     config 1: the four M=126 w8g64 GEMMs with f32 bias, rotated over
            6 distinct weight sets (371 MB > the 256 MB Infinity Cache), as
            achieved HBM GB/s of algorithmic bytes
  i8        config 3: the int8 GEMM at 8160x4096->{4096,16384} on
            pre-quantized operands, TOP/s
  c4        config 4: the 28 linears of one joint audio-video block (20
            launches with the fused QKV / KV packs) over 48 blocks of
            distinct weights, seconds of linear time per denoise step
  roofline  the dominant kernel: at M = 8160 linear_q's default route is the
            dequant-once arm (a 33 us weight expansion, then the dense
            256x256 GEMM), so the GEMM kernel -- timed on its own with HIP
            events on the launch stream, over the expanded weights --
            gives algorithmic FLOP per launch / mean launch time
  cpu_baseline  the reference's CPU linear (oracle/_ref, built from the
            reference's sources) timed on this host, 1 thread, on a row
            sample of the up-projection

  lora      the LoRA delta at the FFN up shape, ranks 32 and 450, and
  dequant_once  the dequant-once A/B arm against the fused kernel there

Usage: python bench.py [--steps K] [--warmup W] [--gpus 1] [--skip-cpu]
                       [--skip-audio] [--skip-i8] [--skip-c4] [--skip-next]
"""
import argparse
import ctypes
import importlib.util
import json
import os
import re
import statistics
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
PEAK_BF16_TFLOPS = 2500.0
PEAK_I8_TOPS = 5000.0
PEAK_HBM_GBS = 8000.0


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def load_package():
    name = "vpipe_ltx25_amd"
    if name in sys.modules:
        return sys.modules[name]
    spec = importlib.util.spec_from_file_location(
        name, os.path.join(ROOT, "vpipe-ltx-2.5_amd", "__init__.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


# ---- synthetic weights, quantized on the GPU ------------------------------------------
def make_qweight(pkg, torch, N, K, gen, std=0.02):
    w = torch.randn((N, K), device="cuda", generator=gen) * std
    codes = torch.empty((N, K), dtype=torch.uint8, device="cuda")
    sc = torch.empty((N, K // 64), dtype=torch.bfloat16, device="cuda")
    qb = torch.empty((N, K // 64), dtype=torch.bfloat16, device="cuda")
    pkg.quantize_affine(w, codes, sc, qb, N, K, 8, 64)
    del w
    return pkg.QWeight(codes, sc, qb, 8, 64)


def gbytes(M, K, N, bias=True):
    """Algorithmic HBM bytes of one w8g64 linear: X + codes + scales/biases
    + Y + f32 bias."""
    return M * K * 2 + N * K + (N * K // 64) * 4 + M * N * 2 + (N * 4 if bias else 0)


class EventTimer:
    """HIP events on torch's current stream, which is the stream the
    library launches on."""

    def __init__(self, torch):
        self.torch = torch
        self.pairs = {}

    def record(self, key, fn):
        t = self.torch
        a = t.cuda.Event(enable_timing=True)
        b = t.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        self.pairs.setdefault(key, []).append((a, b))

    def mean_ms(self, key):
        return float(np.mean([a.elapsed_time(b) for a, b in self.pairs[key]]))

    def total_ms(self, key):
        return float(np.sum([a.elapsed_time(b) for a, b in self.pairs[key]]))


def interleaved(torch, arms, rounds, warmup=3):
    """Best-of-N A/B timing in the reference's manner (tests/ltx25-i8-gemm-test.cc:220-254):
    every round runs each arm once, in an order that alternates between rounds, each call
    bracketed by its own HIP events on the launch stream; the arms therefore see the same
    clock and cache history. Returns {arm: {"best_ms", "median_ms"}}."""
    names = list(arms)
    for _ in range(warmup):
        for n in names:
            arms[n]()
    torch.cuda.synchronize()
    times = {n: [] for n in names}
    for r in range(rounds):
        order = names if r % 2 == 0 else names[::-1]
        evs = []
        for n in order:
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record()
            arms[n]()
            b.record()
            evs.append((n, a, b))
        torch.cuda.synchronize()
        for n, a, b in evs:
            times[n].append(a.elapsed_time(b))
    return {n: {"best_ms": float(min(t)), "median_ms": float(np.median(t))}
            for n, t in times.items()}


def host_description():
    """CPU model and logical CPU count of this host (BASELINE.md asks for both)."""
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        affinity = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        affinity = None
    return {"cpu_model": model, "nproc": os.cpu_count(), "affinity_cpus": affinity}


# ---- config 2: the FFN pair (headline) -------------------------------------------------
def bench_ffn(pkg, torch, steps, warmup, same_tensors=True):
    """The pair through ltx25_linear_q with the library's default routing
    (the dequant-once arm at M = 8160: weight expansion + dense GEMM, both
    inside each timed call). The roofline kernel -- the dense GEMM the route
    runs -- is also timed on its own, on the same stream, over the expanded
    weights: that is the launch the roofline's `achieved` divides by."""
    M, D, H = 8160, 4096, 16384
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    x = torch.randn((M, D), device="cuda", generator=g).to(torch.bfloat16)
    w1 = make_qweight(pkg, torch, H, D, g)
    w2 = make_qweight(pkg, torch, D, H, g)
    h = torch.empty((M, H), dtype=torch.bfloat16, device="cuda")
    y = torch.empty((M, D), dtype=torch.bfloat16, device="cuda")
    route = "dequant-once + dense GEMM" if pkg.dequant_once_takes(M, D, H) else "fused"

    def up():
        pkg.linear_q(x, w1, None, h, M, D, H, pkg.EPI_GELU_TANH)

    def down():
        pkg.linear_q(h, w2, None, y, M, H, D)

    for _ in range(warmup):
        up()
        down()
    # The up / down split comes from a pass of the same steps with events (an
    # event recorded between two launches leaves the GPU idle for about 11 us,
    # rocprof timeline, so the events stay out of the wall-clock pass). It runs
    # before the wall-clock pass: after an idle gap the clock ramps up over
    # the first ~20 steps (2.48, 2.17, 2.24, 2.00, ... ms per step, settling at
    # 1.68-1.70 ms on one box), so with a short warmup the headline's timed
    # steps would otherwise measure the ramp.
    timer = EventTimer(torch)
    for _ in range(steps):
        timer.record("up", up)
        timer.record("down", down)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        up()
        down()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    flop = 2.0 * M * D * H
    up_ms, down_ms = timer.mean_ms("up"), timer.mean_ms("down")
    out = {
        "route": route,
        "ms_per_step": wall / steps * 1e3,
        "tflops": 2 * flop / (wall / steps) / 1e12,
        "up_ms": up_ms,
        "down_ms": down_ms,
        "up_tflops": flop / (up_ms * 1e-3) / 1e12,
        "down_tflops": flop / (down_ms * 1e-3) / 1e12,
        "flop_per_launch": flop,
    }
    # hipBLASLt (torch.matmul on the same bf16 tensors: the dequantized weights this
    # route multiplies, in the same [N][K] layout), and this library's GEMMs over the
    # same dense weights, interleaved best-of-N
    d1 = torch.empty((H, D), dtype=torch.bfloat16, device="cuda")
    d2 = torch.empty((D, H), dtype=torch.bfloat16, device="cuda")
    pkg.dequant(w1, d1, H, D)
    pkg.dequant(w2, d2, D, H)
    c1, c2 = pkg.dense_weight(d1), pkg.dense_weight(d2)
    h_pre = torch.empty_like(h)
    ab = {} if not same_tensors else interleaved(torch, {
        "ours_up_gelu": lambda: pkg.linear_qc(x, c1, None, h, M, D, H, pkg.EPI_GELU_TANH),
        "ours_up": lambda: pkg.linear_qc(x, c1, None, h_pre, M, D, H),
        "hipblaslt_up": lambda: torch.matmul(x, d1.t(), out=h_pre),
        "ours_down": lambda: pkg.linear_qc(h, c2, None, y, M, H, D),
        "hipblaslt_down": lambda: torch.matmul(h, d2.t(), out=y),
    }, rounds=max(10, steps))
    if ab:
        out["same_tensors_vs_hipblaslt"] = {
            k: {"best_us": v["best_ms"] * 1e3, "median_us": v["median_ms"] * 1e3,
                "best_TFLOPs": flop / (v["best_ms"] * 1e-3) / 1e12}
            for k, v in ab.items()}
    if route == "fused":
        out["kernel_mean_ms"] = (up_ms + down_ms) / 2
        return out
    # the route's two kernels, each on its own
    kt = EventTimer(torch)
    for i in range(warmup + steps):
        t = kt if i >= warmup else EventTimer(torch)
        t.record("deq_up", lambda: pkg.dequant(w1, d1, H, D))
        t.record("gemm_up", lambda: pkg.linear_qc(x, c1, None, h, M, D, H, pkg.EPI_GELU_TANH))
        t.record("deq_down", lambda: pkg.dequant(w2, d2, D, H))
        t.record("gemm_down", lambda: pkg.linear_qc(h, c2, None, y, M, H, D))
    torch.cuda.synchronize()
    deq_bytes = H * D * (1 + 2) + (H * D // 64) * 4
    out.update({
        "gemm_up_ms": kt.mean_ms("gemm_up"),
        "gemm_down_ms": kt.mean_ms("gemm_down"),
        "dequant_us": (kt.mean_ms("deq_up") + kt.mean_ms("deq_down")) / 2 * 1e3,
        "dequant_GBps": deq_bytes / ((kt.mean_ms("deq_up") + kt.mean_ms("deq_down")) / 2 * 1e-3)
        / 1e9,
        "kernel_mean_ms": (kt.mean_ms("gemm_up") + kt.mean_ms("gemm_down")) / 2,
    })
    return out


# ---- config 1: audio skinny GEMMs -------------------------------------------------------
AUDIO = [("qkv", 2048, 6144), ("out", 2048, 2048), ("ff_up", 2048, 8192), ("ff_down", 8192, 2048)]


def bench_audio(pkg, torch, steps, warmup, sets=6):
    M = 126
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    xs = {K: torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16) for K in (2048, 8192)}
    weights = []
    for _ in range(sets):
        ws = []
        for name, K, N in AUDIO:
            ws.append((name, K, N, make_qweight(pkg, torch, N, K, g),
                       torch.randn((N,), device="cuda", generator=g) * 0.01,
                       torch.empty((M, N), dtype=torch.bfloat16, device="cuda")))
        weights.append(ws)
    total_weight_mb = sum(N * K * (1 + 4 / 64) for _, K, N in AUDIO) * sets / 1e6

    def one_pass(timer=None):
        for ws in weights:
            for name, K, N, qw, b, yb in ws:
                fn = (lambda K=K, N=N, qw=qw, b=b, yb=yb:
                      pkg.linear_q(xs[K], qw, b, yb, M, K, N))
                if timer is None:
                    fn()
                else:
                    timer.record(name, fn)

    for _ in range(max(1, warmup)):
        one_pass()
    torch.cuda.synchronize()
    timer = EventTimer(torch)
    t0 = time.perf_counter()
    for _ in range(steps):
        one_pass(timer)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    per = {}
    total_bytes = 0.0
    total_ms = 0.0
    for name, K, N in AUDIO:
        ms = timer.mean_ms(name)
        b = gbytes(M, K, N)
        per[name] = {"us": ms * 1e3, "GBps": b / (ms * 1e-3) / 1e9}
        total_bytes += b
        total_ms += ms
    gbs = total_bytes / (total_ms * 1e-3) / 1e9
    # the same GEMMs issued back to back as the block issues them, one event
    # pair around each whole pass over the rotated sets (no per-GEMM events)
    passes = []
    for _ in range(steps):
        a = torch.cuda.Event(enable_timing=True)
        b = torch.cuda.Event(enable_timing=True)
        a.record()
        one_pass()
        b.record()
        passes.append((a, b))
    torch.cuda.synchronize()
    pass_ms = float(np.median([a.elapsed_time(b) for a, b in passes]))
    stream_ms = pass_ms / sets
    # The read ceiling for each GEMM's byte count: the library's own streaming-read probe
    # (ltx25_probe_read: 16-byte loads, four in flight per lane, one workgroup per 16 KB),
    # back to back in a captured burst, its source rotated through a 384 MB pool so that
    # the 256 MB memory-side cache cannot serve repeats.
    reads = read_ceiling(pkg, torch, [(name, gbytes(M, K, N)) for name, K, N in AUDIO], steps)
    return {
        "GBps": gbs,
        "frac_hbm": gbs / PEAK_HBM_GBS,
        "us_four_gemms": total_ms * 1e3,
        "bytes_four_gemms": total_bytes,
        "GBps_back_to_back": total_bytes / (stream_ms * 1e-3) / 1e9,
        "us_four_gemms_back_to_back": stream_ms * 1e3,
        "wall_GBps": total_bytes * sets * steps / wall / 1e9,
        "per_gemm": per,
        "rotated_weight_MB": total_weight_mb,
        "plain_read_same_bytes": reads,
    }


def read_ceiling(pkg, torch, sizes, steps, burst=24):
    """ltx25_probe_read at each (name, bytes), one workgroup per 16 KB (so each byte count
    has a launch shape of its own in a kernel trace), its source rotated through a 384 MB
    pool so that the 256 MB memory-side cache cannot serve repeats. Timed as a captured
    burst of `burst` back-to-back launches over distinct slots (per launch: the replay's
    time / burst; the host's launch cost is out of it), best and median over replays."""
    pool = torch.ones((384 << 20,), dtype=torch.uint8, device="cuda")
    sink = torch.empty((65536,), dtype=torch.int32, device="cuda")
    out = {}
    for name, nbytes in sizes:
        nbytes = (nbytes + 15) // 16 * 16
        span = (nbytes + 4095) // 4096 * 4096
        slots = (pool.numel() - span) // span
        blocks = min(65535, (nbytes + 16383) // 16384)
        views = [pool[(i % slots) * span:] for i in range(burst)]
        for v in views[:4]:
            pkg.probe_read(v, nbytes, sink, blocks)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for v in views:
                pkg.probe_read(v, nbytes, sink, blocks)
        graph.replay()
        torch.cuda.synchronize()
        times = []
        for _ in range(max(10, steps)):
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) / burst)
        del graph
        best, med = min(times), float(np.median(times))
        out[name] = {"bytes": nbytes, "grid": blocks, "best_us": best * 1e3,
                     "best_GBps": nbytes / (best * 1e-3) / 1e9,
                     "median_GBps": nbytes / (med * 1e-3) / 1e9}
    del pool
    return out


def bench_ceilings(pkg, torch, steps):
    """The two ceilings the kernels are measured against, from the library's probes: the
    streaming read at the four C1 GEMMs' and the FFN weight's byte counts, and the MFMA
    stream (16x16x32 bf16, 16384 FLOP each) on zero and random operands at one and two waves
    per SIMD."""
    sizes = [(name, gbytes(126, K, N)) for name, K, N in AUDIO] + [("ffn_weight_codes",
                                                                     16384 * 4096)]
    reads = read_ceiling(pkg, torch, sizes, steps)
    out = torch.empty((256,), dtype=torch.float32, device="cuda")
    iters = 20000
    mfma = {}
    for random in (False, True):
        for wps in (1, 2):
            fn = lambda random=random, wps=wps: pkg.probe_mfma(iters, random, wps, out)
            r = interleaved(torch, {"m": fn}, rounds=max(5, steps // 2))["m"]
            flop = 256.0 * 4 * wps * 8 * iters * 16384
            mfma[f"{'random' if random else 'zero'}_{wps}wave"] = {
                "best_ms": r["best_ms"], "TFLOPs": flop / (r["best_ms"] * 1e-3) / 1e12,
                "frac_bf16_peak": flop / (r["best_ms"] * 1e-3) / 1e12 / PEAK_BF16_TFLOPS}
    return {"read": reads, "mfma_stream": mfma}


# The M <= 128 kernel's phase boundaries, in stamp order (ltx25_probe_skinny_phases)
SKINNY_PHASES = ["codes in registers", "scale block in LDS", "K loop", "partials summed",
                 "stores complete"]
SKINNY_PHASE_CASES = [("qkv", 2048, 6144, 0), ("out", 2048, 2048, 0), ("out", 2048, 2048, 1024),
                      ("out", 2048, 2048, 512), ("ff_up", 2048, 8192, 0),
                      ("ff_down", 8192, 2048, 0)]


def bench_skinny_phases(pkg, torch, steps, sets=6):
    """The audio GEMMs (and the out GEMM forced to 2 and 4 K splits) through the M <= 128
    kernel's phase-stamp instantiation: per case, back-to-back calls over `sets` rotated
    weight sets, the last `sets` calls stamped. Per wave: the time from entry to each phase
    boundary; per call: the span from the first wave's entry to the last wave's end (100 MHz
    clock)."""
    M = 126
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    xs = {K: torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16) for K in (2048, 8192)}
    out = {}
    for name, K, N, k_chunk in SKINNY_PHASE_CASES:
        ws = [(make_qweight(pkg, torch, N, K, g),
               torch.randn((N,), device="cuda", generator=g) * 0.01,
               torch.empty((M, N), dtype=torch.bfloat16, device="cuda")) for _ in range(sets)]
        tiles = (N + 31) // 32
        nwords = 4 * tiles * 8 * 10            # room for 4 splits
        stamps = [torch.zeros((nwords,), dtype=torch.int64, device="cuda") for _ in range(sets)]
        splits = 0

        def call(i):
            qw, b, y = ws[i % sets]
            return pkg.probe_skinny_phases(xs[K], qw, b, y, M, K, N, k_chunk,
                                           stamps[i % sets], nwords * 8)

        for i in range(2 * sets):
            call(i)
        torch.cuda.synchronize()
        for i in range(max(4, steps) * sets):
            splits = call(i)
        torch.cuda.synchronize()
        nwg = splits * tiles
        st = np.stack([s.cpu().numpy()[: nwg * 80].reshape(nwg, 8, 10) for s in stamps])
        clk = st[..., :6].astype(np.float64)
        rt0 = st[..., 6].astype(np.float64)
        rt1 = st[..., 7].astype(np.float64)
        ok = rt1 > rt0
        ghz = float(np.median((clk[..., 5] - clk[..., 0])[ok] / ((rt1 - rt0)[ok] * 10.0)))
        phases = np.diff(clk, axis=-1) / ghz / 1e3                   # us, [call][wg][wave][5]
        span = (rt1.max(axis=(1, 2)) - rt0.min(axis=(1, 2))) * 10.0 / 1e3
        start = (rt0.min(axis=2) - rt0.min(axis=(1, 2))[:, None]) * 10.0 / 1e3   # per WG
        hw = st[..., 0, 8]
        cu = (st[..., 0, 9] & 0xF) * 4096 + ((hw >> 13) & 7) * 256 + ((hw >> 12) & 1) * 16 + \
            ((hw >> 8) & 0xF)
        per_cu = max(int(np.unique(c, return_counts=True)[1].max()) for c in cu)
        out[f"{name} k_chunk={k_chunk or 'plan'}"] = {
            "name": name, "K": K, "N": N, "k_chunk": k_chunk, "splits": splits,
            "workgroups": nwg,
            "clock_GHz": ghz, "span_us_median": float(np.median(span)),
            "wg_start_us_p90": float(np.percentile(start, 90)),
            "max_workgroups_per_cu": per_cu,
            "phase_us_median": {p: float(np.median(phases[..., i]))
                                for i, p in enumerate(SKINNY_PHASES)},
            "phase_us_p90": {p: float(np.percentile(phases[..., i], 90))
                             for i, p in enumerate(SKINNY_PHASES)}}
        del ws, stamps
    return out


TALL_PHASES = ["step 0 landed", "K loop", "output staged", "stores complete"]


def _tall_stamp_stats(st, steps):
    """Stamps [calls][tiles][8 waves][8 words] of the 256 x 256 tile -> per-call spans,
    per-wave phases (us, at each wave's own clock), per-XCD clock and last end, and the gap
    between consecutive tiles on one CU (the next tile's first entry after the last wave of
    the previous one ended)."""
    clk = st[..., :5].astype(np.float64)
    rt0 = st[..., 5].astype(np.float64)
    rt1 = st[..., 6].astype(np.float64)
    ok = rt1 > rt0
    ghz_w = np.where(ok, (clk[..., 4] - clk[..., 0]) / np.maximum((rt1 - rt0) * 10.0, 1.0), np.nan)
    phases = np.diff(clk, axis=-1) / ghz_w[..., None] / 1e3
    xcc = (st[:, :, 0, 7] >> 32) & 0xF
    hw = st[:, :, 0, 7] & 0xFFFFFFFF
    cu = xcc * 4096 + ((hw >> 13) & 7) * 256 + ((hw >> 12) & 1) * 16 + ((hw >> 8) & 0xF)
    base = rt0.min(axis=(1, 2))[:, None]
    start = (rt0.min(axis=2) - base) * 0.01        # us, per call and tile
    end = (rt1.max(axis=2) - base) * 0.01
    gaps = []
    for c in range(st.shape[0]):
        for u in np.unique(cu[c]):
            idx = np.where(cu[c] == u)[0]
            idx = idx[np.argsort(start[c, idx])]
            gaps += [start[c, b] - end[c, a] for a, b in zip(idx[:-1], idx[1:])]
    per_xcc = {}
    for x in range(8):
        m = xcc == x
        if m.any():
            per_xcc[str(x)] = {"tiles_per_call": int(m.sum()) // st.shape[0],
                               "clock_GHz": float(np.nanmedian(ghz_w[m])),
                               "last_end_us": float(np.median([end[c][m[c]].max()
                                                               for c in range(st.shape[0])]))}
    tiles = st.shape[1]
    return {"tiles": tiles, "waves_per_tile": 8, "k_steps": steps,
            "span_us_median": float(np.median(end.max(axis=1))),
            "tile_us_p50_p90": [float(np.percentile(end - start, q)) for q in (50, 90)],
            "tiles_per_cu": sorted({int(v) for v in np.unique(cu[0], return_counts=True)[1]}),
            "gap_us_p50_p90": [float(np.percentile(gaps, q)) for q in (50, 90)] if gaps else None,
            "k_loop_cycles_per_step": float(np.median(clk[..., 2] - clk[..., 1]) / steps),
            "phase_us_median": {p: float(np.nanmedian(phases[..., i]))
                                for i, p in enumerate(TALL_PHASES)},
            "phase_us_p90": {p: float(np.nanpercentile(phases[..., i], 90))
                             for i, p in enumerate(TALL_PHASES)},
            "per_xcc": per_xcc}


def bench_tall_phases(pkg, torch, steps, calls=3):
    """The 256 x 256 tile's phase-stamp instantiation on the config-2 FFN GEMMs (dense bf16
    weights, as the dequant-once route's expansion writes them; up with GELU) and on the
    config-3 int8 GEMM at N = 4096 / 16384: per case, max(20, steps) warm-up calls (the
    clock ramps over the first ~30 ms of MFMA load), then `calls` stamped calls."""
    M, D, H = 8160, 4096, 16384
    g = torch.Generator(device="cuda")
    g.manual_seed(6)
    out = {}
    x = torch.randn((M, D), device="cuda", generator=g).to(torch.bfloat16)
    for name, K, N, epi in (("ffn_up (GELU)", D, H, pkg.EPI_GELU_TANH),
                            ("ffn_down", H, D, pkg.EPI_NONE)):
        xin = x if K == D else torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
        w = (torch.randn((N, K), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        nb = ((M + 255) // 256) * ((N + 255) // 256) * 512
        stamps = [torch.zeros((nb // 8,), dtype=torch.int64, device="cuda") for _ in range(calls)]
        for _ in range(max(20, steps)):
            pkg.probe_tall_phases(xin, w, None, y, M, K, N, epi, stamps[0], nb)
        for s in stamps:
            pkg.probe_tall_phases(xin, w, None, y, M, K, N, epi, s, nb)
        torch.cuda.synchronize()
        st = np.stack([s.cpu().numpy().reshape(-1, 8, 8) for s in stamps]).astype(np.int64)
        out[name] = _tall_stamp_stats(st, K // 64)
        del xin, w, y, stamps
    xq = torch.empty((M, D), dtype=torch.int8, device="cuda")
    sx = torch.empty((M,), dtype=torch.float32, device="cuda")
    pkg.i8_quantize_rows(x, xq, sx, M, D)
    for N in (4096, 16384):
        w = (torch.randn((N, D), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        wq = torch.empty((N, D), dtype=torch.int8, device="cuda")
        sw = torch.empty((N,), dtype=torch.float32, device="cuda")
        pkg.i8_quantize_rows(w, wq, sw, N, D)
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        nb = ((M + 255) // 256) * ((N + 255) // 256) * 512
        stamps = [torch.zeros((nb // 8,), dtype=torch.int64, device="cuda") for _ in range(calls)]
        for _ in range(max(20, steps)):
            pkg.probe_tall_i8_phases(xq, sx, wq, sw, None, y, M, D, N, stamps[0], nb)
        for s in stamps:
            pkg.probe_tall_i8_phases(xq, sx, wq, sw, None, y, M, D, N, s, nb)
        torch.cuda.synchronize()
        st = np.stack([s.cpu().numpy().reshape(-1, 8, 8) for s in stamps]).astype(np.int64)
        out[f"int8 N={N}"] = _tall_stamp_stats(st, D // 128)
        del w, wq, sw, y, stamps
    return out


def tall_phases_summary(json_path, trace_csv, out, cmd):
    """bench.py --tall-phases-only output (stamps) and its rocprofv3 kernel trace (the
    stamped tile's dispatch durations, in case order) -> one markdown file."""
    import csv

    with open(json_path) as f:
        c = json.loads([ln for ln in f.read().splitlines() if ln.startswith("{")][-1])
    c = c["tall_phases"]
    # one case = one run of launches of the stamped tile with no other kernel between them
    runs = []
    with open(trace_csv) as f:
        rows = sorted(csv.DictReader(f), key=lambda r: int(r["Start_Timestamp"]))
    apart = True
    for r in rows:
        name = r["Kernel_Name"].replace("(anonymous namespace)::", "").split("(")[0]
        dur = (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3
        if re.search(r"tall_kernel<\d+, false, true(, \d+)*>$", name):
            if apart:
                runs.append([])
            runs[-1].append(dur)
            apart = False
        else:
            apart = True
    lines = ["# Phase stamps of the 256 x 256 tile (config 2 FFN GEMMs, config 3 int8 GEMM)", "",
             "Commands (MI355X box, repo root):", "", "```", cmd,
             f"python3 bench.py --tall-phases-summary <json> <out>/run_kernel_trace.csv {out} "
             "'<cmd>'", "```", "",
             "`ltx25_probe_tall_phases` / `ltx25_probe_tall_i8_phases` run the same tile as the "
             "routes (M = 8160; the FFN weights dense bf16, as the dequant-once expansion "
             "writes them), instantiated with stamps: lane 0 of each wave reads the shader "
             "clock at entry, when step 0 has landed, after the K loop, after the output tile "
             "is staged in LDS and after its stores complete, and the 100 MHz clock at entry "
             "and end. Three stamped calls per case after the warm-up; phases are medians "
             "(p90) over all waves, each at its own wave's clock. The stamp build waits for its "
             "stores before the last stamp; the product tile does not.", "",
             "| case | tiles | tiles per CU | " + " | ".join(TALL_PHASES) +
             " | tile us p50 / p90 | K-loop cycles per step | span us | rocprof us |",
             "|---|---|---|" + "---|" * len(TALL_PHASES) + "---|---|---|---|"]
    for (key, v), run in zip(c.items(), runs + [None] * len(c)):
        ph = " | ".join(f"{v['phase_us_median'][p]:.2f} ({v['phase_us_p90'][p]:.2f})"
                        for p in TALL_PHASES)
        roc = f"{statistics.median(run[-3:]):.1f}" if run else "-"
        lines.append(f"| {key} | {v['tiles']} | {'/'.join(map(str, v['tiles_per_cu']))} | {ph} | "
                     f"{v['tile_us_p50_p90'][0]:.1f} / {v['tile_us_p50_p90'][1]:.1f} | "
                     f"{v['k_loop_cycles_per_step']:.0f} | {v['span_us_median']:.1f} | {roc} |")
    lines += ["", "Per XCD (clock under load = shader clock ticks per 100 MHz tick; last end = "
              "the XCD's last wave, from the call's first entry):", "",
              "| case | " + " | ".join(f"XCD {x} GHz / last end us" for x in range(8)) + " |",
              "|---|" + "---|" * 8]
    for key, v in c.items():
        cells = [f"{v['per_xcc'][str(x)]['clock_GHz']:.2f} / {v['per_xcc'][str(x)]['last_end_us']:.0f}"
                 if str(x) in v["per_xcc"] else "-" for x in range(8)]
        lines.append(f"| {key} | " + " | ".join(cells) + " |")
    lines += ["", "Gap between consecutive tiles on one CU (us, p50 / p90): " +
              ", ".join(f"{k} {v['gap_us_p50_p90'][0]:.2f} / {v['gap_us_p50_p90'][1]:.2f}"
                        for k, v in c.items() if v["gap_us_p50_p90"]) + "."]
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


def skinny_phases_summary(json_path, trace_csv, out, cmd):
    """bench.py --skinny-phases-only output (stamps) and its rocprofv3 kernel trace (the
    stamped kernels' and their reductions' durations, in case order) -> one markdown file."""
    import csv
    import statistics

    with open(json_path) as f:
        c = json.loads([ln for ln in f.read().splitlines() if ln.startswith("{")][-1])
    c = c["skinny_phases"]
    # One case = one run of launches of the stamped kernel (and their reductions) with no
    # other kernel between them: each case's set-up (its weights) launches kernels first.
    runs = []
    with open(trace_csv) as f:
        rows = sorted(csv.DictReader(f), key=lambda r: int(r["Start_Timestamp"]))
    apart = True
    for r in rows:
        name = r["Kernel_Name"].replace("(anonymous namespace)::", "").split("(")[0]
        dur = (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3
        if re.search(r"skinny_kernel<\d+, (true|false)(, \d+)?, true>$", name):
            key = (int(r.get("Grid_Size_X", r.get("Grid_Size", 0))), int(r.get("Grid_Size_Y", 1)))
            if apart or runs[-1]["key"] != key:
                runs.append({"key": key, "main": [], "reduce": []})
            runs[-1]["main"].append(dur)
            apart = False
        elif "splitk_reduce" in name and runs and not apart:
            runs[-1]["reduce"].append(dur)
        else:
            apart = True
    lines = ["# Phase stamps of the M <= 128 kernel (the audio GEMMs, M = 126, w8g64)", "",
             "Commands (MI355X box, repo root):", "", "```", cmd,
             f"python3 bench.py --skinny-phases-summary <json> <out>/run_kernel_trace.csv {out} "
             "'<cmd>'", "```", "",
             "`ltx25_probe_skinny_phases` runs the same kernel as the linear's M <= 128 route, "
             "instantiated with stamps: lane 0 of each wave reads the shader clock at entry and "
             "at five phase boundaries and the 100 MHz clock at entry and end. Each case runs "
             "over six rotated weight sets, 60 calls after 12 warm-up calls; the last six are "
             "stamped. "
             "Phase times are medians (p90) over all waves of those calls; the span runs from "
             "the first wave's entry to the last wave's end; rocprof is the dispatch's own "
             "duration, which adds launch and drain to the span.", "",
             "| case | splits | workgroups | " + " | ".join(SKINNY_PHASES) +
             " | span us | rocprof main us | rocprof reduce us |",
             "|---|---|---|" + "---|" * len(SKINNY_PHASES) + "---|---|---|"]
    for (key, v), run in zip(c.items(), runs + [None] * len(c)):
        ph = " | ".join(f"{v['phase_us_median'][p]:.2f} ({v['phase_us_p90'][p]:.2f})"
                        for p in SKINNY_PHASES)
        main = f"{statistics.median(run['main']):.2f}" if run else "-"
        red = f"{statistics.median(run['reduce']):.2f}" if run and run["reduce"] else "-"
        lines.append(f"| {key} | {v['splits']} | {v['workgroups']} | {ph} | "
                     f"{v['span_us_median']:.2f} | {main} | {red} |")
    lines += ["", "Clock under load (shader clock ticks per 100 MHz tick): " +
              ", ".join(f"{k} {v['clock_GHz']:.2f} GHz" for k, v in c.items()) + ".",
              "Workgroups per CU at most: " +
              ", ".join(f"{k} {v['max_workgroups_per_cu']}" for k, v in c.items()) + "."]
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


# ---- next rows: the LoRA delta and the dequant-once A/B arm ------------------------------
def bench_lora(pkg, torch, steps, warmup):
    """y += (x . A^T) . B^T at the video FFN shape with the x2 upscaler's rank 32 and the
    distilled adapter's rank 450 (src/ltx25-lora.h): HBM-bound on x and y."""
    M, K, N = 8160, 4096, 16384
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    y = torch.randn((M, N), device="cuda", generator=g).to(torch.bfloat16)
    out = {}
    for rank in (32, 450):
        a = (torch.randn((rank, K), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        b = (torch.randn((N, rank), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        # the reference's signature passes r ([M][rank]) as caller scratch; the r-first
        # route (rank 32 here) computes r into it
        r = torch.empty((M, rank), dtype=torch.bfloat16, device="cuda")
        arms = {"lora": lambda: pkg.lora_add(x, a, b, y, M, K, N, rank),   # noqa: E731
                "lora_caller_r": lambda: pkg.lora_add(x, a, b, y, M, K, N, rank, r=r)}   # noqa: E731
        for fn in arms.values():
            for _ in range(warmup):
                fn()
        timer = EventTimer(torch)
        for _ in range(steps):
            for name, fn in arms.items():
                timer.record(name, fn)
        torch.cuda.synchronize()
        ms = timer.mean_ms("lora")
        byt = M * K * 2 + rank * K * 2 + N * rank * 2 + 2 * M * N * 2
        flop = 2.0 * M * rank * (K + N)
        out[f"rank{rank}"] = {"route": pkg.lora_route(x, a, b, y, M, K, N, rank),
                              "us": ms * 1e3, "caller_r_us": timer.mean_ms("lora_caller_r") * 1e3,
                              "GBps": byt / (ms * 1e-3) / 1e9,
                              "TFLOPs": flop / (ms * 1e-3) / 1e12,
                              "frac_of_linear": None}
    # The adapter on the linear it rides on (the FFN up-projection with GELU, ranks 32 and
    # 450): the linear alone, the linear with the adapter folded into its GEMM
    # (ltx25_linear_q_lora), and the reference's sequence (linear, lora_add, GELU),
    # interleaved best-of-N.
    w = make_qweight(pkg, torch, N, K, g)
    h = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    for rank in (32, 450):
        a = (torch.randn((rank, K), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        b = (torch.randn((N, rank), device="cuda", generator=g) * 0.02).to(torch.bfloat16)

        def seq(a=a, b=b, rank=rank):
            pkg.linear_q(x, w, None, h, M, K, N)
            pkg.lora_add(x, a, b, h, M, K, N, rank)
            pkg.gelu_tanh(h, h)
        ab = interleaved(torch, {
            "linear": lambda: pkg.linear_q(x, w, None, h, M, K, N, pkg.EPI_GELU_TANH),
            "fold": lambda a=a, b=b, rank=rank: pkg.linear_q_lora(x, w, None, a, b, rank, h, M, K,
                                                                  N, pkg.EPI_GELU_TANH),
            "sequence": seq,
        }, rounds=max(10, steps))
        lin = ab["linear"]["best_ms"]
        out[f"rank{rank}_with_linear"] = {
            "fold_taken": pkg.lora_fold_takes(M, K, N, rank, 8),
            # w8 codes, K % 128 == 0 and an aligned A here: merged into the expansion up to
            # rank 64 (ltx25_linear_q_lora's rule), extra K above
            "fold_form": "merged into the expansion" if rank <= 64 else "extra K",
            "linear_us": lin * 1e3,
            "fold_us": ab["fold"]["best_ms"] * 1e3,
            "sequence_us": ab["sequence"]["best_ms"] * 1e3,
            "fold_overhead_frac": ab["fold"]["best_ms"] / lin - 1.0,
            "sequence_overhead_frac": ab["sequence"]["best_ms"] / lin - 1.0,
        }
    return out


def bench_dequant_once(pkg, torch, steps, warmup):
    """The A/B arms at the FFN up-projection (with GELU): the fused dequant-in-GEMM kernel
    against expand-then-dense (the reference's dequant_mma_ route), same shapes, same bits
    out, interleaved best-of-N. Also the int8 tier against the bf16 route at the FFN
    shapes (the tier quantizes X and W per call, inside each timed call)."""
    M, D, H = 8160, 4096, 16384
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = torch.randn((M, D), device="cuda", generator=g).to(torch.bfloat16)
    w = make_qweight(pkg, torch, H, D, g)
    w2 = make_qweight(pkg, torch, D, H, g)
    h = torch.empty((M, H), dtype=torch.bfloat16, device="cuda")
    y = torch.empty((M, D), dtype=torch.bfloat16, device="cuda")
    flop = 2.0 * M * D * H

    def arm(deq=None, i8=False, fn=None):
        def run():
            if deq is not None:
                pkg.set_dequant_once(deq)
            pkg.set_i8_gemm(i8)
            try:
                fn()
            finally:
                pkg.set_dequant_once(pkg.DEQUANT_ONCE_AUTO)
                pkg.set_i8_gemm(False)
        return run

    up = lambda: pkg.linear_q(x, w, None, h, M, D, H, pkg.EPI_GELU_TANH)   # noqa: E731
    down = lambda: pkg.linear_q(h, w2, None, y, M, H, D)                   # noqa: E731
    res = interleaved(torch, {
        "up_fused": arm(pkg.DEQUANT_ONCE_OFF, fn=up),
        "up_dequant_once": arm(pkg.DEQUANT_ONCE_ON, fn=up),
        "up_i8_tier": arm(None, True, up),
        "down_fused": arm(pkg.DEQUANT_ONCE_OFF, fn=down),
        "down_dequant_once": arm(pkg.DEQUANT_ONCE_ON, fn=down),
        "down_i8_tier": arm(None, True, down),
    }, rounds=max(10, steps))
    return {k: {"best_ms": v["best_ms"], "median_ms": v["median_ms"],
                "best_TFLOPs": flop / (v["best_ms"] * 1e-3) / 1e12} for k, v in res.items()}


# ---- config 3: int8 GEMM ----------------------------------------------------------------
def bench_i8(pkg, torch, steps, warmup):
    M, K = 8160, 4096
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    xq = torch.empty((M, K), dtype=torch.int8, device="cuda")
    sx = torch.empty((M,), dtype=torch.float32, device="cuda")
    out = {}
    timer = EventTimer(torch)
    for N in (4096, 16384):
        w = (torch.randn((N, K), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        wq = torch.empty((N, K), dtype=torch.int8, device="cuda")
        sw = torch.empty((N,), dtype=torch.float32, device="cuda")
        pkg.i8_quantize_rows(w, wq, sw, N, K)
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        fn = lambda: pkg.i8_gemm(xq, sx, wq, sw, None, y, None, M, K, N)
        qfn = lambda: pkg.i8_quantize_rows(x, xq, sx, M, K)
        # at least 20 warmup iterations: after the idle gap before the leg the
        # clock ramps up over the first ~30 ms of MFMA load (5 warmup
        # iterations measured 2295 against 2469 TOP/s after 30 at N = 16384)
        for _ in range(max(warmup, 20)):
            qfn()
            fn()
        torch.cuda.synchronize()
        for _ in range(steps):
            timer.record(f"q{N}", qfn)
            timer.record(f"g{N}", fn)
        torch.cuda.synchronize()
        ms = timer.mean_ms(f"g{N}")
        tops = 2.0 * M * K * N / (ms * 1e-3) / 1e12
        out[f"N{N}"] = {"ms": ms, "TOPs": tops, "frac_int8_peak": tops / PEAK_I8_TOPS,
                        "x_quantize_us": timer.mean_ms(f"q{N}") * 1e3}
    return out


# ---- config 4: the linears of 48 joint AV blocks -----------------------------------------
# (name, M, K, N, bias, gelu) per block; M: V video tokens, A audio tokens, T text tokens
BLOCK = [
    ("v_qkv", "V", 4096, 12288, True, False), ("v_out", "V", 4096, 4096, True, False),
    ("v_xq", "V", 4096, 4096, True, False), ("v_xkv", "T", 4096, 8192, True, False),
    ("v_xo", "V", 4096, 4096, True, False), ("v_ff_up", "V", 4096, 16384, False, True),
    ("v_ff_down", "V", 16384, 4096, False, False),
    ("a_qkv", "A", 2048, 6144, True, False), ("a_out", "A", 2048, 2048, True, False),
    ("a_xq", "A", 2048, 2048, True, False), ("a_xkv", "T", 2048, 4096, True, False),
    ("a_xo", "A", 2048, 2048, True, False), ("a_ff_up", "A", 2048, 8192, True, True),
    ("a_ff_down", "A", 8192, 2048, True, False),
    ("a2v_q", "V", 4096, 2048, True, False), ("a2v_kv", "A", 2048, 4096, True, False),
    ("a2v_o", "V", 2048, 4096, True, False),
    ("v2a_q", "A", 2048, 2048, True, False), ("v2a_kv", "V", 4096, 4096, True, False),
    ("v2a_o", "A", 2048, 2048, True, False),
]
TOKENS = {"V": 8160, "A": 126, "T": 1024}


def bench_c4(pkg, torch, steps, warmup, blocks=48):
    """Each block has its own seeded weights AND its own activations (re-seeded per block,
    as BASELINE config 4 states): 48 x ~0.4 GB of inputs plus 19.7 GB of w8g64 weights stay
    resident in HBM."""
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    outs = {}
    for name, mk, K, N, _, _ in BLOCK:
        M = TOKENS[mk]
        if (M, N) not in outs:
            outs[(M, N)] = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    stack = []
    params = 0
    for blk_i in range(blocks):
        ga = torch.Generator(device="cuda")
        ga.manual_seed(1000 + blk_i)
        acts = {}
        blk = []
        for name, mk, K, N, has_bias, gelu in BLOCK:
            M = TOKENS[mk]
            if (M, K) not in acts:
                acts[(M, K)] = torch.randn((M, K), device="cuda", generator=ga).to(torch.bfloat16)
            qw = make_qweight(pkg, torch, N, K, g)
            b = torch.randn((N,), device="cuda", generator=g) * 0.01 if has_bias else None
            blk.append((acts[(M, K)], M, K, N, qw, b, gelu))
            params += N * K
        stack.append(blk)
    flop_block = sum(2.0 * TOKENS[mk] * K * N for _, mk, K, N, _, _ in BLOCK)

    def step():
        for blk in stack:
            for xa, M, K, N, qw, b, gelu in blk:
                pkg.linear_q(xa, qw, b, outs[(M, N)], M, K, N,
                             pkg.EPI_GELU_TANH if gelu else pkg.EPI_NONE)

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    s = (time.perf_counter() - t0) / steps
    # block 0's launches timed one at a time after the timed region (HIP events on the launch
    # stream, median of 10 after 2), with the route each took: a badly routed shape shows here
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    per_launch = {}
    for (name, _, _, _, _, _), (xa, M, K, N, qw, b, gelu) in zip(BLOCK, stack[0]):
        ts = []
        for r in range(12):
            ev0.record()
            pkg.linear_q(xa, qw, b, outs[(M, N)], M, K, N,
                         pkg.EPI_GELU_TANH if gelu else pkg.EPI_NONE)
            ev1.record()
            torch.cuda.synchronize()
            if r >= 2:
                ts.append(ev0.elapsed_time(ev1) * 1e3)
        us = statistics.median(ts)
        route = pkg.linear_route(M, K, N, 8)
        per_launch[name] = {"M": M, "K": K, "N": N, "us": round(us, 1),
                            "tflops": round(2.0 * M * K * N / us / 1e6, 1),
                            "tile": route["tile"], "dequant_once": route["dequant_once"],
                            "splits": route["splits"]}
    return {"s_per_denoise_step": s, "tflops": flop_block * blocks / s / 1e12,
            "flop_per_block": flop_block, "params": params, "blocks": blocks,
            "launches_per_block": len(BLOCK), "timed_steps": steps, "warmup_steps": warmup,
            "activations": "re-seeded per block (seeds 1000..1047)",
            "block0_launches_us_sum": round(sum(v["us"] for v in per_launch.values()), 1),
            "block0_per_launch": per_launch}


# ---- CPU baseline -------------------------------------------------------------------------
def cpu_baseline(c2_rows=128, c3_rows=256):
    """The CPU path on this host, per config, each
    figure with its seconds and threads:
      - c0, c1: the reference's CPU linear (oracle/_ref: src/ltx25-block-ref.cc:11-28
        compiled from the reference sources; the oracle's restatement of the
        same loop, "port", where oracle/_ref was not built) over the weight
        dequantized by the oracle's restatement of the reference quantizer,
        run fully: C0 320 x 4096 -> 4096 with an f32 bias, the four C1 audio
        GEMMs at 126 tokens with bias (GB/s of the algorithmic bytes, the
        metric config 1 is quoted in);
      - c2: the same linear on a row sample of the up-projection 8160 x 4096
        -> 16384 (the headline; the rate scales linearly with rows), and the
        oracle's OpenMP f32 port on all threads;
      - c3: the oracle's exact int32 GEMM (orc_i8_gemm_i32) on a row sample
        of the int8 tier at 8160 x 4096 -> 4096.
    The top-level value is the c2 rate (the headline's unit and workload)."""
    orc_path = os.path.join(ROOT, "oracle", "liboracle.so")
    ref_path = os.path.join(ROOT, "oracle", "_ref", "libltx25ref.so")
    if not os.path.exists(orc_path):
        return None
    o = ctypes.CDLL(orc_path)
    vp, ci = ctypes.c_void_p, ctypes.c_int
    o.orc_fill_normal.argtypes = [vp, ctypes.c_size_t, ctypes.c_uint64, ctypes.c_float, ctypes.c_float]
    o.orc_quantize_affine.argtypes = [vp, ci, ci, ci, ci, vp, vp, vp, vp]
    o.orc_dequant.argtypes = [vp, vp, vp, ci, ci, ci, ci, vp, vp]
    o.orc_linear_f64.argtypes = [vp, vp, vp, ci, ci, ci, vp]
    o.orc_linear_f32_omp.argtypes = [vp, vp, vp, ci, ci, ci, vp, ci]
    o.orc_i8_gemm_i32.argtypes = [vp, vp, ci, ci, ci, vp]
    kind = "port"
    lin = o.orc_linear_f64
    if os.path.exists(ref_path):
        r = ctypes.CDLL(ref_path)
        r.ref_linear.argtypes = [vp, vp, vp, ci, ci, ci, vp]
        lin = r.ref_linear
        kind = "reference"

    def normal(shape, seed, std):
        a = np.empty(shape, np.float32)
        o.orc_fill_normal(a.ctypes.data, a.size, seed, 0.0, std)
        return a

    def dequantized(N, K, seed):
        """N(0, 0.02) weights through the reference quantizer, dequantized to f32."""
        w = normal((N, K), seed, 0.02)
        codes = np.empty((N, K // 4), np.uint32)
        sc = np.empty((N, K // 64), np.uint16)
        qb = np.empty((N, K // 64), np.uint16)
        o.orc_quantize_affine(w.ctypes.data, N, K, 8, 64, codes.ctypes.data, sc.ctypes.data,
                              qb.ctypes.data, None)
        o.orc_dequant(codes.ctypes.data, sc.ctypes.data, qb.ctypes.data, N, K, 8, 64,
                      w.ctypes.data, None)
        return w

    def timed_linear(M, K, N, seed, bias=True):
        w = dequantized(N, K, seed)
        x = normal((M, K), seed + 1, 1.0)
        b = normal((N,), seed + 2, 0.01) if bias else None
        out = np.empty((M, N), np.float32)
        t0 = time.perf_counter()
        lin(x.ctypes.data, w.ctypes.data, None if b is None else b.ctypes.data, M, K, N,
            out.ctypes.data)
        return time.perf_counter() - t0, x, w, out

    host = host_description()
    res = {"host": host, "kind": kind, "cores": 1}
    # C0, fully
    t, *_ = timed_linear(320, 4096, 4096, 11)
    res["c0"] = {"value": 2.0 * 320 * 4096 * 4096 / t / 1e12, "unit": "TFLOP/s", "seconds": t,
                 "cores": 1, "kind": kind,
                 "sample": "all of config 0: 320 x 4096 -> 4096 w8g64 (dequantized to f32) + f32 "
                           "bias, double accumulator, 1 thread"}
    # C1, fully
    t1 = 0.0
    per = {}
    for i, (name, K, N) in enumerate(AUDIO):
        t, *_ = timed_linear(126, K, N, 21 + 3 * i)
        per[name] = {"seconds": t, "GBps": gbytes(126, K, N) / t / 1e9}
        t1 += t
    c1_bytes = sum(gbytes(126, K, N) for _, K, N in AUDIO)
    res["c1"] = {"value": c1_bytes / t1 / 1e9, "unit": "GB/s", "seconds": t1, "cores": 1,
                 "kind": kind, "per_gemm": per,
                 "sample": "all four config-1 audio GEMMs at 126 tokens with bias, back to "
                           "back, double accumulator, 1 thread"}
    # C2, row sample of the up-projection
    D, H = 4096, 16384
    t, x, w, out = timed_linear(c2_rows, D, H, 7, bias=False)
    flop = 2.0 * c2_rows * D * H
    threads = min(16, os.cpu_count() or 1)
    t_omp0 = time.perf_counter()
    o.orc_linear_f32_omp(x.ctypes.data, w.ctypes.data, None, c2_rows, D, H, out.ctypes.data,
                         threads)
    t_omp = time.perf_counter() - t_omp0
    res["c2"] = {"value": flop / t / 1e12, "unit": "TFLOP/s", "seconds": t, "cores": 1,
                 "kind": kind,
                 "sample": (f"{c2_rows} of 8160 rows of the config-2 up-projection 4096->16384 "
                            f"(w8g64 dequantized to f32), double accumulator, 1 thread; the rate "
                            f"scales linearly to all rows"),
                 "omp_f32": {"value": flop / t_omp / 1e12, "unit": "TFLOP/s", "cores": threads,
                             "kind": "port", "seconds": t_omp}}
    del x, w, out
    # C3, row sample of the int8 GEMM (exact int32)
    K3, N3 = 4096, 4096
    rng = np.random.default_rng(31)
    xq = rng.integers(-127, 128, size=(c3_rows, K3), dtype=np.int8)
    wq = rng.integers(-127, 128, size=(N3, K3), dtype=np.int8)
    acc = np.empty((c3_rows, N3), np.int32)
    t0 = time.perf_counter()
    o.orc_i8_gemm_i32(xq.ctypes.data, wq.ctypes.data, c3_rows, K3, N3, acc.ctypes.data)
    t3 = time.perf_counter() - t0
    res["c3"] = {"value": 2.0 * c3_rows * K3 * N3 / t3 / 1e12, "unit": "TOP/s", "seconds": t3,
                 "cores": 1, "kind": "port",
                 "sample": f"{c3_rows} of 8160 rows of the config-3 int8 GEMM 4096->4096, exact "
                           f"int32 accumulation (the oracle's loop), 1 thread"}
    res.update({
        "value": res["c2"]["value"],
        "unit": "TFLOP/s",
        "sample": res["c2"]["sample"] + " (per-config figures under c0..c3)",
        "omp_f32": res["c2"]["omp_f32"],
    })
    return res


TRAFFIC_JSON = os.path.join(ROOT, "profiles", "qgemm_ffn_hbm_traffic.json")
COPY_BYTES = 256 << 20   # the --profile-copy kernel reads and writes this much


def load_traffic():
    if os.path.exists(TRAFFIC_JSON):
        with open(TRAFFIC_JSON) as f:
            return json.load(f)
    return None


# The roofline kernel's launches by rocprofv3 (kernel trace of the FFN leg
# without the same-tensor comparison, so every launch of the kernel at the
# two FFN shapes is the route's own): written by --kernel-grid-summary,
# read back into the bench line beside the HIP-event figure.
ROOF_JSON = os.path.join(ROOT, "profiles", "roofline_kernel_stats.json")
ROOF_MD = os.path.join(ROOT, "profiles", "roofline_kernel_stats.md")  # the one summary that writes it
FFN_GRIDS = {((8160 + 255) // 256) * (16384 // 256) * 512: "up",
             ((8160 + 255) // 256) * (4096 // 256) * 512: "down"}


def load_roof():
    if os.path.exists(ROOF_JSON):
        with open(ROOF_JSON) as f:
            return json.load(f)
    return None


def tall_mode(name):
    """The operand mode of a tall.hip launch (0 dense bf16, 1 int8, 2 fused w8) read from its
    kernel name (`tall_kernel<0>` or `tall_kernel<0, false>`; the fused w8 tile is
    `tall_w8_kernel`), else None."""
    import re

    if "tall_w8_kernel" in name:
        return 2
    m = re.search(r"tall_kernel<(\d)[,>]", name)
    return int(m.group(1)) if m else None


def _pmc_rows(path):
    import csv

    out = {}
    with open(path) as f:
        for r in csv.DictReader(f):
            out[int(r["Dispatch_Id"])] = (r["Kernel_Name"], int(r["Grid_Size"]),
                                          float(r["Counter_Value"]))
    return out


def pmc_summary(fetch_csv, write_csv, cmd):
    """HBM traffic per launch from two rocprofv3 --pmc runs of the same bench
    command (FETCH_SIZE, then WRITE_SIZE; both KiB per dispatch), each scaled
    by what the counter reads for the plain 256 MiB device copy that
    --profile-copy adds (the last copy dispatch). Writes the markdown summary
    and the JSON that the roofline's `traffic` field reads."""
    fe, wr = _pmc_rows(fetch_csv), _pmc_rows(write_csv)
    copies = [i for i, (n, _, _) in fe.items() if "copyBuffer" in n or "copy_kernel" in n]
    big = [i for i in copies if fe[i][2] > 1000 and wr.get(i, ("", 0, 0))[2] > 1000]
    if not big:
        raise SystemExit("no calibration copy in the counter files (run with --profile-copy)")
    cal = max(big)
    f_fac = COPY_BYTES / (fe[cal][2] * 1024)
    w_fac = COPY_BYTES / (wr[cal][2] * 1024)
    groups = {}
    for i, (name, grid, v) in fe.items():
        if "Cijk_" in name:
            short = "hipBLASLt " + name    # the same-tensor comparison leg
        elif ("qgemm_kernel" not in name and "tall_kernel" not in name and
                "tall_w8_kernel" not in name and "splitk_reduce" not in name and
                "dequant_kernel" not in name):
            continue
        else:
            short = name[name.index("ltx25::"):].split("(ltx25")[0].replace("(anonymous namespace)::", "")
        g = groups.setdefault((short, grid), [0, 0.0, 0.0])
        g[0] += 1
        g[1] += v * 1024 * f_fac
        g[2] += wr.get(i, ("", 0, 0.0))[2] * 1024 * w_fac
    M, D, H = 8160, 4096, 16384

    def alg(which, dense):
        """read, write bytes of an FFN GEMM: w8g64 codes + scales/biases, or the bf16
        expansion the dequant-once route's dense GEMM reads."""
        k, n = (D, H) if which == "up" else (H, D)
        w = n * k * 2 if dense else n * k + n * k // 64 * 4
        return (M * k * 2 + w, M * n * 2)

    mt = (M + 255) // 256
    ffn_grid = {mt * (H // 256) * 512: "up", mt * (D // 256) * 512: "down"}
    lines = ["# HBM traffic per launch (rocprofv3 FETCH_SIZE / WRITE_SIZE)", "",
             "Commands (two counter runs of the same program, then this summary):", "",
             "```", cmd, "```", "",
             f"Calibration: the 256 MiB device copy (dispatch {cal}) reads "
             f"{fe[cal][2]:.0f} KiB by FETCH_SIZE and writes {wr[cal][2]:.0f} KiB by WRITE_SIZE, "
             f"so FETCH_SIZE is scaled by {f_fac:.3f} and WRITE_SIZE by {w_fac:.3f}.", "",
             "| kernel | grid | launches | fetch MB/launch | write MB/launch | algorithmic read / write MB |",
             "|---|---|---|---|---|---|"]
    ffn = []
    for (short, grid), (n, fb, wb) in sorted(groups.items(), key=lambda kv: -kv[1][1] / kv[1][0]):
        if short.startswith("hipBLASLt"):
            lines.append(f"| `{short}` | {grid} | {n} | {fb / n / 1e6:.1f} | {wb / n / 1e6:.1f} | "
                         f"up and down mixed (the same tensors as the dense GEMM) |")
            continue
        # the 256 x 256 tile of tall.hip: mode 0 dense bf16, 2 fused w8 dequant
        tall_dense = tall_mode(short) == 0
        tall_fused = tall_mode(short) == 2
        which = ffn_grid.get(grid) if "256, 256" in short or tall_dense or tall_fused else None
        dense = ", 16, " in short or tall_dense
        a = (f"{alg(which, dense)[0] / 1e6:.1f} / {alg(which, dense)[1] / 1e6:.1f} ({which})"
             if which else "")
        lines.append(f"| `{short}` | {grid} | {n} | {fb / n / 1e6:.1f} | {wb / n / 1e6:.1f} | {a} |")
        if which:
            ffn.append(((fb + wb) / n, which, dense))
    # the roofline kernel: the dense GEMM when the route ran it, else the fused one
    if any(d for _, _, d in ffn):
        ffn = [f for f in ffn if f[2]]
    traffic = sum(t for t, _, _ in ffn) / len(ffn) if ffn else None
    alg_mean = sum(sum(alg(w, d)) for _, w, d in ffn) / len(ffn) if ffn else None
    lines += ["", f"FFN GEMM (the roofline kernel, mean of up and down): "
              f"{traffic / 1e6:.1f} MB per launch against {alg_mean / 1e6:.1f} MB algorithmic."
              if traffic else "", ""]
    with open(os.path.join(ROOT, "profiles", "qgemm_ffn_hbm_traffic.md"), "w") as f:
        f.write("\n".join(lines))
    with open(TRAFFIC_JSON, "w") as f:
        json.dump({"traffic_bytes": round(traffic) if traffic else None,
                   "algorithmic_bytes": round(alg_mean) if alg_mean else None,
                   "fetch_factor": round(f_fac, 4), "write_factor": round(w_fac, 4),
                   "source": "profiles/qgemm_ffn_hbm_traffic.md"}, f, indent=1)
    print("\n".join(lines))


def busy_summary(csv_path, out, cmd):
    """Shader clock, MFMA-busy and L2-busy per kernel from one rocprofv3 --pmc
    run with GRBM_GUI_ACTIVE, SQ_VALU_MFMA_BUSY_CYCLES and TCC_BUSY_avr, and,
    when the run also counted them, the fraction of wave cycles spent waiting
    on any instruction dependency (SQ_WAIT_INST_ANY / SQ_WAVE_CYCLES) and on
    LDS instruction issue (SQ_WAIT_INST_LDS / SQ_WAVE_CYCLES), and the LDS
    bank-conflict cycles per launch (SQ_LDS_BANK_CONFLICT, summed over CUs).
    GRBM_GUI_ACTIVE counts the graphics engine's active cycles summed over
    the 8 XCDs, so /8 / duration is the clock; SQ_VALU_MFMA_BUSY_CYCLES sums
    the busy cycles of every SIMD (32 per v_mfma_f32_32x32x16_bf16, 16 per
    v_mfma_f32_16x16x32_bf16), so
    dividing by the SIMD count (4 per CU) x the active cycles gives the
    fraction of the elapsed time the matrix cores ran; TCC_BUSY_avr is the
    mean busy cycles of an L2 channel."""
    import csv

    xcds, simds = 8, 4 * 256
    per = {}
    with open(csv_path) as f:
        for r in csv.DictReader(f):
            name = r["Kernel_Name"]
            if "ltx25::" in name:
                short = name[name.index("ltx25::"):].replace("(anonymous namespace)::", "")
                short = short.split("(")[0]
            elif "Cijk_" in name:
                short = "hipBLASLt " + name    # the same-tensor comparison leg
            else:
                continue
            key = (short, int(r["Grid_Size"]))
            d = per.setdefault(key, {"dur": {}, "c": {}})
            i = int(r["Dispatch_Id"])
            d["dur"][i] = int(r["End_Timestamp"]) - int(r["Start_Timestamp"])
            d["c"].setdefault(r["Counter_Name"], {})[i] = float(r["Counter_Value"])
    lines = ["# Clock, MFMA-busy and L2-busy per kernel (rocprofv3 --pmc)", "", "Command:", "",
             "```", cmd, "```", "",
             f"clock = GRBM_GUI_ACTIVE / {xcds} XCDs / duration; MFMA busy = "
             f"SQ_VALU_MFMA_BUSY_CYCLES / ({simds} SIMDs x active cycles); L2 busy = "
             "TCC_BUSY_avr / active cycles. Durations are the profiled dispatches' own. The "
             "ratios mean something only for dispatches of ~100 us and more: the counters of "
             "a short one also cover its launch and drain (hence clocks above the 2.4 GHz "
             "maximum).", "",
             "| kernel | grid | launches | avg us | clock GHz | MFMA busy | L2 busy | "
             "wait any | wait LDS issue | LDS conflict cycles |",
             "|---|---|---|---|---|---|---|---|---|---|"]
    for (short, grid), d in sorted(per.items(), key=lambda kv: -sum(kv[1]["dur"].values())):
        ids = sorted(d["dur"])
        g = d["c"].get("GRBM_GUI_ACTIVE", {})
        mb = d["c"].get("SQ_VALU_MFMA_BUSY_CYCLES", {})
        tb = d["c"].get("TCC_BUSY_avr", {})
        dur = sum(d["dur"][i] for i in ids) / len(ids)
        cyc = sum(g.get(i, 0.0) for i in ids) / len(ids) / xcds
        mf = sum(mb.get(i, 0.0) for i in ids) / len(ids)
        l2 = sum(tb.get(i, 0.0) for i in ids) / len(ids)
        clk = cyc / dur if dur else 0.0

        def mean(c):
            v = d["c"].get(c, {})
            return sum(v.get(i, 0.0) for i in ids) / len(ids) if v else None

        wc, wa, wl, bc = (mean(c) for c in ("SQ_WAVE_CYCLES", "SQ_WAIT_INST_ANY",
                                            "SQ_WAIT_INST_LDS", "SQ_LDS_BANK_CONFLICT"))
        frac = lambda a: f"{a / wc:.2f}" if a is not None and wc else "-"
        lines.append(f"| `{short}` | {grid} | {len(ids)} | {dur / 1e3:.1f} | {clk:.2f} | "
                     f"{mf / (simds * cyc) if cyc else 0:.2f} | {l2 / cyc if cyc else 0:.2f} | "
                     f"{frac(wa)} | {frac(wl)} | {f'{bc:.3g}' if bc is not None else '-'} |")
    lines.append("")
    with open(out, "w") as f:
        f.write("\n".join(lines))
    print("\n".join(lines))


def kernel_summary(db, out, cmd, note):
    """rocprofv3 kernel-trace database -> a short markdown table (via rocpd2summary)."""
    import csv
    import subprocess
    import tempfile

    d = tempfile.mkdtemp()
    subprocess.run(["rocpd2summary", "-i", os.path.abspath(db), "-f", "csv", "-d", d, "-o", "k"],
                   cwd="/tmp", check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(os.path.join(d, "k_kernels_summary.csv")) as f:
        rows = list(csv.DictReader(f))
    lines = [f"# Kernel stats: {note}", "", "Commands (MI355X box, repo root):", "", "```", cmd,
             f"python3 bench.py --kernel-summary <out>/run_results.db {out} '<cmd>' '<note>'",
             "```", "", "| kernel | calls | avg us | min us | max us | total % |",
             "|---|---|---|---|---|---|"]
    for r in rows:
        n = r["Name"]
        n = n if len(n) <= 100 else n[:100] + "..."
        lines.append(f"| `{n}` | {r['Calls']} | {float(r['Average (Nsec)']) / 1e3:.1f} | "
                     f"{float(r['Min (Nsec)']) / 1e3:.1f} | {float(r['Max (Nsec)']) / 1e3:.1f} | "
                     f"{float(r['Percent (Inc)']):.1f} |")
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


def kernel_grid_summary(trace_csv, out, cmd, note):
    """rocprofv3 kernel_trace.csv -> markdown per (kernel, grid): one row per
    launch shape, so the four audio GEMMs and the plain reads of their byte
    counts read separately."""
    import csv
    import statistics

    groups = {}
    with open(trace_csv) as f:
        for r in csv.DictReader(f):
            name = r["Kernel_Name"].replace("(anonymous namespace)::", "")
            name = name.split("(")[0] if "(" in name else name
            name = name if len(name) <= 90 else name[:90] + "..."
            key = (name, int(r.get("Grid_Size", r.get("Grid_Size_X", 0))))
            groups.setdefault(key, []).append(
                (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3)
    lines = [f"# Kernel stats per launch shape: {note}", "", "Commands (MI355X box, repo root):",
             "", "```", cmd,
             f"python3 bench.py --kernel-grid-summary <out>/run_kernel_trace.csv {out} '<cmd>' "
             "'<note>'", "```", "",
             "| kernel | grid (threads) | calls | median us | mean us | min us |",
             "|---|---|---|---|---|---|"]
    for (name, grid), v in sorted(groups.items(), key=lambda kv: -sum(kv[1])):
        if len(v) < 4:
            continue
        lines.append(f"| `{name}` | {grid} | {len(v)} | {statistics.median(v):.1f} | "
                     f"{statistics.mean(v):.1f} | {min(v):.1f} |")
    # the roofline kernel (tall_kernel<0> at the two FFN grids), when traced for the roofline
    # summary (other traces, e.g. the audio leg's, also hold FFN launches)
    ffn = {FFN_GRIDS[g]: statistics.mean(v) for (n, g), v in groups.items()
           if tall_mode(n) == 0 and g in FFN_GRIDS}
    if len(ffn) == 2 and os.path.basename(out) == os.path.basename(ROOF_MD):
        mean_us = (ffn["up"] + ffn["down"]) / 2
        flop = 2.0 * 8160 * 4096 * 16384
        tf = flop / (mean_us * 1e-6) / 1e12
        lines += ["", f"Roofline kernel (`tall_kernel<0>`, mean of the up and down means): "
                  f"{mean_us:.1f} us per launch = {tf:.1f} TFLOP/s = "
                  f"{tf / PEAK_BF16_TFLOPS:.4f} of the bf16 peak."]
        with open(ROOF_JSON, "w") as f:
            json.dump({"up_us": round(ffn["up"], 2), "down_us": round(ffn["down"], 2),
                       "mean_us": round(mean_us, 2), "tflops": round(tf, 2),
                       "frac": round(tf / PEAK_BF16_TFLOPS, 4),
                       "source": os.path.relpath(out, ROOT)}, f, indent=1)
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


def ceilings_summary(json_path, trace_csv, out, cmd):
    """bench.py --ceilings-only output (the rates) and its rocprofv3 kernel trace (the probe
    kernels' own durations) -> one markdown summary."""
    import csv
    import statistics

    with open(json_path) as f:
        c = json.loads([ln for ln in f.read().splitlines() if ln.startswith("{")][-1])["ceilings"]
    groups = {}
    with open(trace_csv) as f:
        for r in csv.DictReader(f):
            name = r["Kernel_Name"].replace("(anonymous namespace)::", "").split("(")[0]
            if "probe" not in name and "stream" not in name:
                continue
            key = (name, int(r.get("Grid_Size", r.get("Grid_Size_X", 0))))
            groups.setdefault(key, []).append(
                (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3)
    lines = ["# The library's own ceilings: streaming read and MFMA stream", "",
             "Commands (MI355X box, repo root):", "", "```", cmd,
             f"python3 bench.py --ceilings-summary <json> <out>/run_kernel_trace.csv {out} '<cmd>'",
             "```", "",
             "Streaming read (`ltx25_probe_read`: 16-byte non-temporal loads, one workgroup per "
             "16 KB, one word per workgroup to a sink, rotated over a 384 MB pool so no launch "
             "reads what the last one did; per launch = a captured burst of 24 back-to-back "
             "launches / 24, best and median of the replays):", "",
             "| bytes of | bytes | grid (workgroups) | best us | best GB/s | median GB/s |",
             "|---|---|---|---|---|---|"]
    for name, v in c["read"].items():
        lines.append(f"| {name} | {v['bytes']} | {v['grid']} | {v['best_us']:.2f} | "
                     f"{v['best_GBps']:.0f} | {v['median_GBps']:.0f} |")
    lines += ["", "MFMA stream (`ltx25_probe_mfma`: v_mfma_f32_16x16x32_bf16 back to back on 8 "
              "accumulators, 256 workgroups, zero or xorshift-random bf16 operands):", "",
              "| operands, waves per SIMD | best ms | TFLOP/s | fraction of the 2.5 PFLOP/s peak |",
              "|---|---|---|---|"]
    for name, v in c["mfma_stream"].items():
        lines.append(f"| {name} | {v['best_ms']:.3f} | {v['TFLOPs']:.0f} | "
                     f"{v['frac_bf16_peak']:.3f} |")
    lines += ["", "Probe kernels in the trace:", "",
              "| kernel | grid (threads) | calls | median us | min us |", "|---|---|---|---|---|"]
    for (name, grid), v in sorted(groups.items()):
        lines.append(f"| `{name}` | {grid} | {len(v)} | {statistics.median(v):.2f} | "
                     f"{min(v):.2f} |")
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("\n".join(lines))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    # 30 FFN steps (about 55 ms of sustained load) before the timed ones: with
    # 3, the first timed steps still ran below the settled clock (1207 vs
    # 1261 TFLOP/s for the same kernels, the event-timed split agreeing with
    # the latter).
    ap.add_argument("--warmup", type=int, default=30,
                    help="untimed steps before the timed ones (default 30)")
    ap.add_argument("--skip-cpu", action="store_true")
    ap.add_argument("--skip-audio", action="store_true")
    ap.add_argument("--skip-i8", action="store_true")
    ap.add_argument("--skip-c4", action="store_true")
    ap.add_argument("--skip-hipblaslt", action="store_true",
                    help="skip the FFN leg's same-tensor comparison with hipBLASLt (for a kernel "
                         "trace whose launches of the roofline kernel are all the route's own)")
    ap.add_argument("--skip-next", action="store_true",
                    help="skip the LoRA-delta and dequant-once measurements")
    ap.add_argument("--ceilings", action="store_true",
                    help="also measure the library's ceiling probes (streaming read at the audio "
                         "GEMMs' byte counts, MFMA stream on zero and random operands)")
    ap.add_argument("--ceilings-only", action="store_true",
                    help="measure only the ceiling probes and print them as one JSON line")
    ap.add_argument("--profile-copy", action="store_true",
                    help="also run one plain 256 MiB device copy, the known-size kernel that "
                         "calibrates rocprofv3 FETCH_SIZE / WRITE_SIZE")
    ap.add_argument("--kernel-grid-summary", nargs=4, metavar=("TRACE_CSV", "OUT_MD", "CMD", "NOTE"),
                    help="write a per-launch-shape kernel table from a rocprofv3 kernel trace")
    ap.add_argument("--pmc-summary", nargs=3, metavar=("FETCH_CSV", "WRITE_CSV", "CMD"),
                    help="summarise two rocprofv3 --pmc counter files into profiles/ and exit")
    ap.add_argument("--kernel-summary", nargs=4, metavar=("DB", "OUT_MD", "CMD", "NOTE"),
                    help="summarise a rocprofv3 --kernel-trace database into OUT_MD and exit")
    ap.add_argument("--busy-summary", nargs=3, metavar=("CSV", "OUT_MD", "CMD"),
                    help="summarise a rocprofv3 --pmc run of GRBM_GUI_ACTIVE, "
                         "SQ_VALU_MFMA_BUSY_CYCLES and TCC_BUSY_avr into OUT_MD and exit")
    ap.add_argument("--ceilings-summary", nargs=4, metavar=("JSON", "TRACE_CSV", "OUT_MD", "CMD"),
                    help="summarise a --ceilings-only run and its rocprofv3 kernel trace into "
                         "OUT_MD and exit")
    ap.add_argument("--tall-phases-only", action="store_true",
                    help="run only the 256 x 256 tile's phase-stamp probes (FFN GEMMs, int8 "
                         "GEMM) and print the stamps' statistics as one JSON line")
    ap.add_argument("--tall-phases-summary", nargs=4,
                    metavar=("JSON", "TRACE_CSV", "OUT_MD", "CMD"),
                    help="summarise a --tall-phases-only run and its rocprofv3 kernel trace "
                         "into OUT_MD and exit")
    ap.add_argument("--skinny-phases-only", action="store_true",
                    help="run only the M <= 128 kernel's phase-stamp probe over the audio GEMMs "
                         "and print the stamps as one JSON line")
    ap.add_argument("--skinny-phases-summary", nargs=4,
                    metavar=("JSON", "TRACE_CSV", "OUT_MD", "CMD"),
                    help="summarise a --skinny-phases-only run and its rocprofv3 kernel trace "
                         "into OUT_MD and exit")
    args = ap.parse_args()
    if args.ceilings_summary:
        ceilings_summary(*args.ceilings_summary)
        return
    if args.skinny_phases_summary:
        skinny_phases_summary(*args.skinny_phases_summary)
        return
    if args.tall_phases_summary:
        tall_phases_summary(*args.tall_phases_summary)
        return
    if args.busy_summary:
        busy_summary(*args.busy_summary)
        return
    if args.kernel_summary:
        kernel_summary(*args.kernel_summary)
        return
    if args.kernel_grid_summary:
        kernel_grid_summary(*args.kernel_grid_summary)
        return
    if args.pmc_summary:
        pmc_summary(*args.pmc_summary)
        return
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py measures one GPU: this build's path runs on a single MI355X; "
              "the multi-GPU sharding is designed but not built. Run with --gpus 1.",
              file=sys.stderr)
        sys.exit(2)

    import torch

    pkg = load_package()
    pkg.load()
    torch.cuda.set_device(0)
    pkg.check(pkg.load().ltx25_init())

    if args.ceilings_only:
        print(json.dumps({"ceilings": bench_ceilings(pkg, torch, args.steps)}), flush=True)
        return
    if args.tall_phases_only:
        print(json.dumps({"tall_phases": bench_tall_phases(pkg, torch, args.steps)}), flush=True)
        return
    if args.skinny_phases_only:
        print(json.dumps({"skinny_phases": bench_skinny_phases(pkg, torch, args.steps)}),
              flush=True)
        return
    log(f"FFN pair (config 2): warmup {args.warmup}, steps {args.steps}")
    ffn = bench_ffn(pkg, torch, args.steps, args.warmup, same_tensors=not args.skip_hipblaslt)
    log(f"  {ffn['tflops']:.1f} TFLOP/s, up {ffn['up_ms']:.3f} ms, down {ffn['down_ms']:.3f} ms")
    torch.cuda.empty_cache()
    extra = {}
    if not args.skip_audio:
        log("audio (config 1)")
        extra["audio"] = bench_audio(pkg, torch, max(5, args.steps // 2), args.warmup)
        log(f"  {extra['audio']['GBps']:.0f} GB/s per-GEMM events, "
            f"{extra['audio']['GBps_back_to_back']:.0f} GB/s back to back")
        torch.cuda.empty_cache()
    if not args.skip_i8:
        log("int8 (config 3)")
        extra["i8"] = bench_i8(pkg, torch, args.steps, args.warmup)
        log(f"  {extra['i8']}")
        torch.cuda.empty_cache()
    if not args.skip_next:
        log("LoRA delta and the dequant-once arm")
        extra["lora"] = bench_lora(pkg, torch, max(5, args.steps // 2), args.warmup)
        ffn_ms = ffn["up_ms"]
        for v in extra["lora"].values():
            if "us" in v:
                v["frac_of_linear"] = v["us"] * 1e-3 / ffn_ms
        extra["ab_interleaved"] = bench_dequant_once(pkg, torch, max(5, args.steps // 2),
                                                     args.warmup)
        log(f"  {extra['lora']}\n  {extra['ab_interleaved']}")
        torch.cuda.empty_cache()
    if args.ceilings:
        log("ceiling probes")
        extra["ceilings"] = bench_ceilings(pkg, torch, args.steps)
        torch.cuda.empty_cache()
    if not args.skip_c4:
        log("48-block linear set (config 4)")
        extra["c4"] = bench_c4(pkg, torch, steps=5, warmup=2)
        log(f"  {extra['c4']['s_per_denoise_step']:.3f} s/step")
        torch.cuda.empty_cache()
    if args.profile_copy:
        src = torch.ones((256 << 20,), dtype=torch.uint8, device="cuda")
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    cpu = None
    if not args.skip_cpu:
        log("CPU baseline")
        cpu = cpu_baseline()
        if cpu:
            log(f"  {cpu['value']*1e3:.3f} GFLOP/s ({cpu['kind']})")

    achieved = ffn["flop_per_launch"] / (ffn["kernel_mean_ms"] * 1e-3) / 1e12
    traffic = load_traffic()
    roof = load_roof()
    line = {
        "metric": "qlinear TFLOP/s + % MFMA peak at M=8160 K=4096 N=16384 w8g64; audio GB/s",
        "value": round(ffn["tflops"], 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ffn["ms_per_step"], 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: X ~ N(0,1) bf16, W ~ N(0,0.02) quantized w8g64 on the GPU, seeded",
        "config": {"workload": "config 2: video FFN pair 8160x4096->16384 (GELU-tanh fused) "
                               "->4096, w8g64, no bias",
                   "M": 8160, "K": 4096, "N": 16384, "quant": "w8g64"},
        "pct_bf16_peak": round(100 * ffn["tflops"] / PEAK_BF16_TFLOPS, 2),
        "ffn": {k: (round(v, 4) if isinstance(v, float) else v) for k, v in ffn.items()},
        "roofline": {
            "kernel": ("tall_kernel<0> (the 256x256 dense bf16 GEMM on 16x16x32 MFMAs, "
                       "dequant-once route; up with GELU and down)" if ffn["route"] != "fused" else
                       "tall_kernel<2> (the 256x256 tile, w8 codes dequantized in registers; "
                       "up with GELU and down)"),
            "bound": "mfma",
            "achieved": round(achieved, 2),
            "peak": PEAK_BF16_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(achieved / PEAK_BF16_TFLOPS, 4),
            "traffic": traffic.get("traffic_bytes") if traffic else None,
            # the same kernel's mean launch time by rocprofv3 (committed profile)
            "rocprof_mean_us": roof.get("mean_us") if roof else None,
            "frac_rocprof": roof.get("frac") if roof else None,
        },
        "cpu_baseline": cpu,
    }
    line.update(extra)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
