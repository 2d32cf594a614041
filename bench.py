"""Benchmark of the escape-time render path on one MI355X.

Workload (one step): the 4096x4096 plain-Mandelbrot frame at centre
(-0.743643887037151, 0.131825904205330), real-axis width 1e-4, 4 seeded-jitter
samples per pixel, maxIter 5000, bailout |z|^2 >= 256, rendered in FP64 with the
reference's rounding (bit-exact escape counts) by the straggler-compaction frame
pipeline, with the smooth value and the RGBA8 colour through a 256-entry palette.
Inputs (tile descriptors, palette) are resident on the device before timing.
value = Giga-iterations/s over the timed steps, in iterations of the reference's
loop: an interior sample counts maxIter, also where the kernels find its orbit to be a
cycle and stop.  In this frame they run 99.5 % of the iterations counted; in frames with
much of the set's interior (the deep frames, the uneven batch, the 1024x1024 frame) far
fewer, so that rates and FLOP rates there are what the reference's loop would have to
reach and may exceed what the hardware can issue.

Also reported (variants): the reference's CPU-runnable 1024x1024 frame (maxIter
1000) on the GPU (the CPU-baseline leg runs it in full through the oracle on the
host and compares the counts), the 256-tile uneven batch (autotuned, captured
replay), 16 zoom sessions through the continuous-batching loop (p50/p99
arrival-to-completion latency), the drop-in FractalRenderer path at 3840x2160
(renderQuality and renderFast), the 1920x1080 deep-zoom frames (FP32 and FP64-delta perturbation and
direct FP64 with their mismatch against the double-double oracle subset and their
algorithmic FLOP rate against the FP32 / FP64 vector peak: 15 FLOPs per
perturbation step, 8 per direct step, whole frame including the reference orbit), and
the roofline of the dominant kernel (pass 1 of the pipeline:
8 algorithmic FP64 FLOPs per iteration it executes, against the 78.6 TFLOP/s
FP64 vector peak, and its iteration rate against the issue ceiling of the fused
step's 6 FP64 VALU instructions: 39.3e12 lane-instructions/s / 6), the thread-per-
sample grid kernel and the FP32 pipeline on the same frame, and the oracle's CPU
rate on a bounded row band of the same frame on the host's cores.

python bench.py [--steps K] [--warmup W] [--gpus 1] [--no-cpu] [--no-variants]
                [--leg c1|uneven|deep|serving|serving_capacity|renderer]
"""
from __future__ import annotations

import argparse
import ctypes
import importlib
import json
import os
import re
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Giga-iter/s (FP32 perturb vs FP64 direct, % vector peak); p50/p99 frame ms"
COUNTED = ("iterations of the reference's loop; interior orbits found to be cycles stop early, so "
           "rates of frames with interior may exceed the issue ceiling")
CENTER = (-0.743643887037151, 0.131825904205330)
W = H = 4096
SPP = 4
MAX_ITER = 5000
BAILOUT_SQ = 256.0
SEED = 20261202
FLOPS_PER_ITER = 8
# a perturbation step: (2Z + d) d + dc as 6 FMAs (12 FLOPs) and the rebase test
# fma(Zx, dx, Zy * dy) < -|Z|^2/2 (a product and an FMA, 3 FLOPs)
PERTURB_FLOPS_PER_ITER = 15
FP64_PEAK_TFLOPS = 78.6
# the fused FP64 step issues 6 VALU instructions (3 mul, 2 add, 1 fma); FP64
# instructions issue at 16 lanes per cycle per SIMD = FP64_PEAK_TFLOPS / 2 lane-ops/s
FP64_ISSUE_CEILING_GITER = FP64_PEAK_TFLOPS / 2 * 1e3 / 6
FP32_PEAK_TFLOPS = 157.3
# block_steps, handoff_lanes, tail_passes, drain_refill: pass 1 hands its
# stragglers to one persistent drain launch that refills lanes once 40 wait
TUNE = (16, 24, 0, 40)
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "c2_fp64_pass1_traffic.md")


def frame_tune(cu, tune):
    """cu.FrameTune (wave shape 0) from (block_steps, handoff_lanes, tail_passes, drain_refill)."""
    b, h, p, d = tune
    return cu.FrameTune(b, h, p, 0, d)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def frame_tile(cu):
    seg = cu.plane_segment_from_center(CENTER[0], CENTER[1], 1e-4, W, H)
    return cu.make_tile(*seg, W, H, MAX_ITER, BAILOUT_SQ, spp=SPP, pattern=cu.SAMPLE_JITTER,
                        seed=SEED)


def palette(cu):
    pal = ((np.arange(256, dtype=np.uint32) * 0x00010305) | 0xFF000000).astype(np.uint32)
    return cu.DeviceBuffer.from_array(pal)


class PipelineRun:
    """One frame object of the pipeline; each step renders it with compose."""

    def __init__(self, cu, engine, tile, precision, tune):
        self.cu = cu
        self.frame = cu.Frame(engine, [tile], precision, -1)
        self.tune = frame_tune(cu, tune)
        self.pal = palette(cu)
        self.rgba = cu.DeviceBuffer(tile.width * tile.height * 4)
        self.pass1_ms, self.total_ms = [], []

    def step(self):
        self.frame.render(self.tune, self.pal, 256, self.rgba)
        p1, tot = self.frame.last_ms()
        self.pass1_ms.append(p1)
        self.total_ms.append(tot)

    def reset(self):
        self.pass1_ms, self.total_ms = [], []

    def iterations(self):
        return self.frame.iterations(), self.frame.iterations_pass1()

    def close(self):
        self.frame.close()


class GridRun:
    """Thread-per-sample grid kernel (escape_tile) plus the separate compose."""

    def __init__(self, cu, engine, tile, precision):
        self.cu, self.engine, self.tile, self.precision = cu, engine, tile, precision
        n = tile.width * tile.height
        self.counts = cu.DeviceBuffer(n * 4)
        self.smooth = cu.DeviceBuffer(n * 8)
        self.rgba = cu.DeviceBuffer(n * 4)
        self.iters = cu.IterationCounter()
        self.pal = palette(cu)
        self.variant = 1 if cu.tile_fused_safe(tile, precision) else 0
        self.pass1_ms, self.total_ms = [], []

    def step(self):
        t = self.tile
        self.engine.escape_tile(self.precision, t, self.counts, self.smooth, self.iters, self.variant)
        self.pass1_ms.append(self.engine.last_kernel_ms())
        self.total_ms.append(self.pass1_ms[-1])
        self.engine.compose_smooth(self.smooth, t.width, self.rgba, t.width, t.width, t.height,
                                   self.pal, 256)

    def reset(self):
        self.pass1_ms, self.total_ms = [], []
        self.iters.clear()

    def iterations(self):
        it = self.iters.total()
        return it, it

    def close(self):
        pass


def timed(cu, run, steps: int, warmup: int):
    """Warm up, then time exactly `steps` steps between two device synchronisations.
    Returns (seconds, iterations per step, pass-1 iterations per step)."""
    for _ in range(warmup):
        run.step()
    cu.synchronize()
    run.reset()
    t0 = time.perf_counter()
    for _ in range(steps):
        run.step()
    cu.synchronize()
    dt = time.perf_counter() - t0
    total, first = run.iterations()
    if isinstance(run, GridRun):  # the grid counter accumulates over the timed steps
        total, first = total // steps, first // steps
    return dt, total, first


def uneven_leg(cu, engine):
    """The 256-tile uneven batch: default pipeline tune vs the autotuner's pick."""
    wl = importlib.import_module("chaos-ultra_amd.workloads")
    at = importlib.import_module("chaos-ultra_amd.autotune")
    t0 = time.perf_counter()
    tiles, info = wl.uneven_tiles(cu, 256)
    gen_s = time.perf_counter() - t0
    res = at.tune_batch(cu, engine, tiles, repeats=3, warmup=1)
    frame = cu.Frame(engine, tiles, 64, -1)
    out = {"tiles": len(tiles), "pixels": int(sum(i["side"] ** 2 for i in info)),
           "generate_s": round(gen_s, 1)}
    for name, tn in (("default", cu.FrameTune(16, 16, 5, 0)),
                     ("tuned_pipeline", at.frame_tune(cu, res["pipeline"]["best"]))):
        ms = []
        for _ in range(4):
            frame.render(tn)
            ms.append(frame.last_ms()[1])
        it = frame.iterations()
        m = float(np.median(ms[1:]))
        out[name] = {"render_ms": round(m, 3), "giga_iter_s": round(it / m / 1e6, 1),
                     "iterations": int(it)}
    frame.capture(tn)
    ms = []
    for _ in range(4):
        frame.replay()
        ms.append(frame.last_ms()[1])
    out["tuned_pipeline"]["graph_replay_ms"] = round(float(np.median(ms[1:])), 3)
    frame.close()
    if res["engine"] == "persistent":  # time the winner on its own
        batch = at.PersistentBatch(cu, tiles)
        p = res["tune"]
        tn = cu.Tune(p["block_steps"], p["waves_per_cu"], p["chunk"], p["refill_lanes"])
        ms = [batch.render(engine, tn) for _ in range(4)]
        it = batch.iters.total()
        m = float(np.median(ms[1:]))
        out["tuned_persistent"] = {"render_ms": round(m, 3), "giga_iter_s": round(it / m / 1e6, 1),
                                   "iterations": int(it)}
        # the winner as one captured launch (clears and kernel in a HIP graph)
        g = batch.capture(engine, tn)
        gms = []
        for _ in range(4):
            g.replay()
            gms.append(g.last_ms())
        g.close()
        gm = float(np.median(gms[1:]))
        out["tuned_persistent"]["graph_replay_ms"] = round(gm, 3)
        out["tuned_persistent"]["graph_replay_giga_iter_s"] = round(batch.iters.total() / gm / 1e6, 1)
    out["autotune"] = {"engine": res["engine"], "tune": res["tune"], "ms": round(res["ms"], 3),
                       "pipeline_best": res["pipeline"]["best"],
                       "persistent_best": res.get("persistent", {}).get("best"),
                       "persistent_ms": round(res.get("persistent", {}).get("ms", float("nan")), 3),
                       "candidates": len(res["pipeline"]["table"]) +
                                     len(res.get("persistent", {}).get("table", []))}
    return out


def smooth_error(got, want, same):
    """Relative smooth-value error |got - want| / max(|want|, 1) over the pixels whose
    counts agree (`same`): p50, p99 and max."""
    rel = np.abs(got - want) / np.maximum(np.abs(want), 1.0)
    r = rel[same]
    if r.size == 0:
        return None
    return {"p50": float(np.percentile(r, 50)), "p99": float(np.percentile(r, 99)),
            "max": float(r.max()), "pixels": int(r.size)}


def deep_leg(cu, engine):
    """1920x1080 deep-zoom frames (maxIter 50000): FP64/FP32-delta perturbation and
    direct FP64; rate, mismatch and smooth-value error against direct FP64 on the
    full frame (at 1e-6 and 1e-10, where direct FP64 resolves the pixels) and
    against the committed double-double subset (all widths)."""
    g = np.load(os.path.join(ROOT, "tests", "golden", "deep_dd_subset.npz"))
    idx = g["index"]
    out = {}
    for w in (1e-6, 1e-10, 1e-20):
        row = {}
        planes = {}
        dd_c = g[f"counts_{w:.0e}"].astype(np.uint32)
        dd_s = g[f"smooth_{w:.0e}"].astype(np.float64)
        for name, method in (("perturb_f64", cu.DEEP_PERTURB_F64), ("perturb_f32", cu.DEEP_PERTURB_F32),
                             ("direct_f64", cu.DEEP_DIRECT_F64)):
            if method == cu.DEEP_DIRECT_F64 and w < 1e-13:
                continue  # below the FP64 ulp of the centre
            d = cu.make_deep(-0.743643887037151, 0.131825904205330, w, 1920, 1080, 50000, 256.0)
            f = cu.DeepFrame(engine, d, method)
            ms = []
            for _ in range(3):
                f.render()
                ms.append(f.report().total_ms)
            rep = f.report()
            full_c, full_s = f.counts().ravel(), f.smooth().ravel()
            planes[name] = (full_c, full_s)
            counts, smooth = full_c[idx], full_s[idx]
            f.close()
            m = float(np.median(ms))
            flops = PERTURB_FLOPS_PER_ITER if method != cu.DEEP_DIRECT_F64 else FLOPS_PER_ITER
            peak = FP32_PEAK_TFLOPS if method == cu.DEEP_PERTURB_F32 else FP64_PEAK_TFLOPS
            tflops = rep.iterations * flops / (m * 1e-3) / 1e12
            row[name] = {"frame_ms": round(m, 3), "giga_iter_s": round(rep.iterations / m / 1e6, 1),
                         "tflops": round(tflops, 2), "frac_of_vector_peak": round(tflops / peak, 4),
                         "mismatch_vs_dd_pct": round(100 * float(np.mean(counts != dd_c)), 3),
                         "smooth_rel_err_vs_dd": smooth_error(smooth, dd_s, counts == dd_c)}
            if method != cu.DEEP_DIRECT_F64:
                row[name]["orbit_ms"] = round(rep.orbit_ms, 3)
                # a zoom sequence toward the same centre keeps the orbit between frames
                d.flags = cu.DEEP_REBASE | cu.DEEP_REUSE_ORBIT
                f = cu.DeepFrame(engine, d, method)
                kept = []
                for _ in range(3):
                    f.render()
                    kept.append(f.report().total_ms)
                f.close()
                row[name]["frame_ms_orbit_kept"] = round(float(np.median(kept[1:])), 3)
        if "direct_f64" in row:
            row["perturb_f32_over_direct_f64"] = round(row["perturb_f32"]["giga_iter_s"] /
                                                       row["direct_f64"]["giga_iter_s"], 3)
            dc, ds = planes["direct_f64"]
            for name in ("perturb_f64", "perturb_f32"):
                c, sm = planes[name]
                row[name]["mismatch_vs_direct_f64_pct"] = round(100 * float(np.mean(c != dc)), 3)
                row[name]["smooth_rel_err_vs_direct_f64"] = smooth_error(sm, ds, c == dc)
        out[f"width_{w:.0e}"] = row
    return out


def renderer_leg(cu, w=3840, h=2160, frames=5):
    """The drop-in path (FractalRenderer): renderQuality on the module's default
    view (supplyDefaultValues: centre (-0.5, 0), zoom 2, maxIterations 1600,
    maxSuperSampling 5, adaptive) at 3840x2160, then renderFast frames zooming in
    by 0.977 about the centre with reuse and foveation, then renderQuality at the
    frame pipeline's view (FP64 by the precision switch, maxIter 5000) with 1, 4
    and 16 (adaptive) samples.  Iterations are the module's executed-iteration
    count (cu_renderer_iterations)."""
    prov = cu.FractalRendererProvider()
    r = prov.get_default_renderer()
    try:
        r.initialize_rendering(w, h, cu.default_palette())
        m = cu.RenderingModel()
        r.supply_default_values(m, w, h)
        m.use_adaptive_super_sampling = 1
        m.use_sample_reuse = 1
        m.use_foveated_rendering = 1
        r.render_quality(m)  # warm-up
        out = {"view": "default (centre -0.5,0; zoom 2)", "size": f"{w}x{h}",
               "max_iter": int(m.max_iterations), "max_super_sampling": float(m.max_super_sampling)}
        ms, its = [], []
        for _ in range(frames):
            i0, t0 = r.iterations(), time.perf_counter()
            r.render_quality(m)
            ms.append((time.perf_counter() - t0) * 1e3)
            its.append(r.iterations() - i0)
        k = int(np.argsort(ms)[len(ms) // 2])
        out["render_quality"] = {"ms_p50": round(ms[k], 3), "iterations": int(its[k]),
                                 "giga_iter_s": round(its[k] / ms[k] / 1e6, 1)}
        ms, its = [], []
        cx = 0.5 * (m.left_bottom_x + m.right_top_x)
        cy = 0.5 * (m.left_bottom_y + m.right_top_y)
        for _ in range(frames * 4):
            hw = 0.5 * (m.right_top_x - m.left_bottom_x) * 0.977
            hh = 0.5 * (m.right_top_y - m.left_bottom_y) * 0.977
            m.set_segment(cx - hw, cy - hh, cx + hw, cy + hh)
            m.zooming, m.zooming_in = 1, 1
            m.mouse_focus_x, m.mouse_focus_y = w // 2, h // 2
            i0, t0 = r.iterations(), time.perf_counter()
            r.render_fast(m)
            ms.append((time.perf_counter() - t0) * 1e3)
            its.append(r.iterations() - i0)
        out["render_fast"] = {"frames": len(ms), "ms_p50": round(float(np.median(ms)), 3),
                              "giga_iter_s": round(float(np.sum(its)) / float(np.sum(ms)) / 1e6, 1)}
        # the frame pipeline's view (C2 centre, width 1e-4) at 4K through renderQuality: the
        # precision switch picks the FP64 kernel (pixel 2.6e-8 below the float ulp of 0.74)
        seg = cu.plane_segment_from_center(CENTER[0], CENTER[1], 1e-4 * h / w, w, h)
        out["c2_view_fp64"] = {}
        for max_ss, adaptive in ((1.0, 0), (4.0, 0), (16.0, 1)):
            m = cu.RenderingModel()
            r.supply_default_values(m, w, h)
            m.set_segment(*seg)
            m.max_iterations = MAX_ITER
            m.max_super_sampling = max_ss
            m.use_adaptive_super_sampling = adaptive
            m.use_sample_reuse = 0
            m.use_foveated_rendering = 0
            r.render_quality(m)  # warm-up
            ms, its = [], []
            for _ in range(frames):
                i0, t0 = r.iterations(), time.perf_counter()
                r.render_quality(m)
                ms.append((time.perf_counter() - t0) * 1e3)
                its.append(r.iterations() - i0)
            k = int(np.argsort(ms)[len(ms) // 2])
            out["c2_view_fp64"][f"max_ss_{max_ss:g}{'_adaptive' if adaptive else ''}"] = {
                "ms_p50": round(ms[k], 3), "iterations": int(its[k]),
                "giga_iter_s": round(its[k] / ms[k] / 1e6, 1),
                "precision": "fp64" if m.floating_point_precision == cu.PRECISION_DOUBLE else "fp32"}
        r.free_rendering_resources()
        return out
    finally:
        prov.close()


def serving_leg(cu, hbm_budget=16 << 30, slots=8):
    """16 zoom sessions, Poisson arrivals at 30 fps each, 120 frames, replayed in
    real time through the continuous-batching loop."""
    sv = importlib.import_module("chaos-ultra_amd.serve")
    sessions = sv.zoom_sessions(16, 120)
    server = sv.Server(cu.KERNELS_DIR, hbm_budget, slots=slots)
    try:
        recs, span = sv.run(server, sessions, realtime=True)
        out = sv.summarise(recs, sessions, server.report(), span)
    finally:
        server.close()
    out.update({"hbm_budget_bytes": hbm_budget, "slots": slots, "deep_method": "fp32 perturbation",
                "start_widths": "log-uniform in [1e-14, 3]; frames below 1e-12 use perturbation",
                "resolutions": [f"{s['width']}x{s['height']}" for s in sessions]})
    return out


def serving_capacity_leg(cu, frames=45, p99_target_ms=33.0, slots=8, hbm_budget=192 << 30,
                         seed=20261203):
    """How many 3840x2160 zoom sessions one GPU serves at 30 frames/s with the p99
    arrival -> completion latency within p99_target_ms: sessions drawn as in the
    serving leg but all at 4K, replayed in real time; the session count doubles from
    8 until the p99 exceeds the target, then bisects between the last two counts."""
    sv = importlib.import_module("chaos-ultra_amd.serve")

    def run_n(n):
        sessions = sv.zoom_sessions(n, frames, seed=seed, resolutions=((3840, 2160),))
        server = sv.Server(cu.KERNELS_DIR, hbm_budget, slots=slots)
        try:
            recs, span = sv.run(server, sessions, realtime=True, timeout_s=120.0)
            s = sv.summarise(recs, sessions, server.report(), span)
        finally:
            server.close()
        log(f"[bench] serving capacity: {n} 4K sessions -> p50 {s['p50_ms']} ms, p99 {s['p99_ms']} ms, "
            f"{s['giga_iter_s']} G-iter/s")
        return {k: s[k] for k in ("p50_ms", "p99_ms", "max_ms", "giga_iter_s", "frames",
                                  "frames_reuse", "frames_full", "frames_deep", "peak_bytes")}

    runs = {}
    ok, n = 0, 8
    while n <= 512:
        runs[n] = run_n(n)
        if runs[n]["p99_ms"] > p99_target_ms:
            break
        ok, n = n, n * 2
    lo, hi = ok, n
    while hi - lo > max(1, lo // 8):
        mid = (lo + hi) // 2
        runs[mid] = run_n(mid)
        if runs[mid]["p99_ms"] <= p99_target_ms:
            lo = mid
        else:
            hi = mid
    return {"sustainable_4k_sessions_at_30fps": lo, "p99_target_ms": p99_target_ms,
            "frames_per_session": frames, "slots": slots, "hbm_budget_bytes": hbm_budget,
            "shallow_precision": "fp64", "deep_method": "fp32 perturbation below width 1e-12",
            "runs": {str(k): runs[k] for k in sorted(runs)}}


def read_traffic():
    """HBM bytes per pass-1 launch from the committed counter summary, if present."""
    try:
        with open(TRAFFIC_FILE) as f:
            m = re.search(r"traffic_bytes_per_launch:\s*([0-9]+)", f.read())
        return int(m.group(1)) if m else None
    except OSError:
        return None


def cpu_baseline(cu, tile, gpu_counts=None, gpu_smooth=None, c1=None, seconds_target=15.0):
    """The oracle (a scalar C++ restatement of the reference iteration, OpenMP over rows)
    on a bounded row band of the same frame.  The band's counts and smooth values are
    compared with the same rows of the GPU's frame (gpu_counts / gpu_smooth, the
    full 4096x4096 planes of the timed render).  With c1 = (tile, pipeline counts,
    grid-kernel counts) of the 1024x1024 frame, that frame also runs in full through
    the oracle and its counts are compared with both GPU engines'."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import _oracle
    threads = os.cpu_count() or 1
    try:
        threads = len(os.sched_getaffinity(0))
    except AttributeError:
        pass
    r0 = H // 2  # probe 4 rows to size the sample, then time a band of rows around the centre
    t0 = time.perf_counter()
    _oracle.escape_tile(tile, 64, rows=(r0, r0 + 4), threads=threads)
    probe = max(time.perf_counter() - t0, 1e-3)
    rows = int(max(4, min(H, 4 * seconds_target / 3 / probe)))
    a = max(0, r0 - rows // 2)
    rates, it, dts = [], 0, []
    for _ in range(3):  # median of 3 runs of the band
        t0 = time.perf_counter()
        band_c, band_s, it = _oracle.escape_tile(tile, 64, rows=(a, a + rows), threads=threads)
        dts.append(time.perf_counter() - t0)
        rates.append(it / dts[-1] / 1e9)
    check = {}
    if gpu_counts is not None:
        g_c = gpu_counts.reshape(H, W)[a:a + rows]
        g_s = gpu_smooth.reshape(H, W)[a:a + rows]
        o_c, o_s = band_c[a:a + rows], band_s[a:a + rows]
        rel = np.abs(g_s - o_s) / np.maximum(np.abs(o_s), 1.0)
        check = {"same_counts": bool(np.array_equal(g_c, o_c)),
                 "pixels_compared": int(g_c.size),
                 "smooth_max_rel_diff": float(rel.max()),
                 "smooth_within_1e-12": bool(rel.max() <= 1e-12)}
    cpu_model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    cpu_model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    c1_check = {}
    if c1 is not None:
        c1_tile, c1_pipe, c1_grid = c1
        c1_dts = []
        for _ in range(3):
            t0 = time.perf_counter()
            want, _, cit = _oracle.escape_tile(c1_tile, 64, threads=threads)
            c1_dts.append(time.perf_counter() - t0)
        c1_check = {"ms_p50": round(float(np.median(c1_dts)) * 1e3, 2),
                    "giga_iter_s": round(cit / float(np.median(c1_dts)) / 1e9, 3),
                    "threads": threads,
                    "same_counts": bool(np.array_equal(c1_pipe, want) and
                                        np.array_equal(c1_grid, want))}
    return {"value": round(float(np.median(rates)), 4), "unit": "Giga-iter/s", "cores": threads,
            "cpu_model": cpu_model, "kind": "port",
            "sample": f"rows {a}..{a + rows - 1} of the 4096x4096 FP64 frame (4 spp, maxIter 5000), "
                      f"{it} iterations per run, median of 3 runs ({', '.join(f'{d:.2f}' for d in dts)} s); "
                      f"g++ -O2 -ffp-contract=off, OpenMP {threads} threads",
            **({"vs_gpu_frame": check} if check else {}),
            **({"c1_frame_in_full": c1_check} if c1_check else {})}


def c1_leg(cu, engine):
    """The reference's CPU-runnable case: the 1024x1024 FP64 frame, centre (-0.5, 0),
    width 3, 1 sample at each pixel centre, maxIter 1000, bailout 4 (counts and
    smooth values), through the frame pipeline and through the one-launch grid
    kernel.  The headline figures are the faster engine's: 97 % of
    this frame's iterations belong to the 17 % of its pixels inside the set, which
    run all 1000 steps; the pipeline hands them on to its drain launch, while the
    grid kernel runs them to the end in place.  Returns the JSON entry and the
    tile with the pipeline's counts, for the CPU baseline leg's full-frame check."""
    tile = cu.make_tile(-2.0, -1.5, 1.0, 1.5, 1024, 1024, 1000, 4.0)
    fr = cu.Frame(engine, [tile], 64, -1)
    tn = frame_tune(cu, TUNE)
    for _ in range(3):
        fr.render(tn)
    ms = []
    for _ in range(20):
        fr.render(tn)
        ms.append(fr.last_ms()[1])
    it = fr.iterations()
    counts = fr.counts()
    fr.close()
    pipe_ms = float(np.median(ms))

    n = tile.width * tile.height
    g_counts, g_smooth = cu.DeviceBuffer(n * 4), cu.DeviceBuffer(n * 8)
    g_iters = cu.IterationCounter()
    variant = 1 if cu.tile_fused_safe(tile, 64) else 0
    gms = []
    for k in range(23):
        g_iters.clear()
        engine.escape_tile(64, tile, g_counts, g_smooth, g_iters, variant)
        if k >= 3:
            gms.append(engine.last_kernel_ms())
    git = g_iters.total()
    gcounts = g_counts.download(np.uint32, n)
    for b in (g_counts, g_smooth, g_iters):
        b.close()
    grid_ms = float(np.median(gms))

    best_ms, engine_name = (grid_ms, "grid") if grid_ms < pipe_ms else (pipe_ms, "pipeline")
    out = {"iterations": it, "engine": engine_name, "render_ms_p50": round(best_ms, 4),
           "giga_iter_s": round(it / best_ms / 1e6, 1),
           "pipeline": {"render_ms_p50": round(pipe_ms, 4), "giga_iter_s": round(it / pipe_ms / 1e6, 1),
                        "tune": list(TUNE)},
           "grid_kernel": {"kernel_ms_p50": round(grid_ms, 4), "giga_iter_s": round(git / grid_ms / 1e6, 1),
                           "iterations": git, "same_counts_as_pipeline": bool(np.array_equal(gcounts, counts))}}
    return out, (tile, counts.reshape(1024, 1024), gcounts.reshape(1024, 1024))


def calibrate_copy(cu, mib):
    """A device-to-device copy of `mib` MiB: a plain copy of known size that scales the
    FETCH_SIZE / WRITE_SIZE counters."""
    if not mib:
        return
    n = mib << 20
    src, dst = cu.DeviceBuffer(n), cu.DeviceBuffer(n)
    src.fill_u32(1)
    cu.abi.call("cu_memcpy_dtod", dst.ptr, src.ptr, n)
    cu.synchronize()
    log(f"[bench] copied {mib} MiB device-to-device for counter calibration")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-variants", action="store_true",
                    help="skip the grid / FP32 variants and the uneven-tile and deep-zoom legs")
    ap.add_argument("--leg", choices=["all", "c1", "uneven", "deep", "serving", "serving_capacity",
                                      "renderer"],
                    default="all",
                    help="run one leg only and print its JSON (used for profiling)")
    ap.add_argument("--calibrate-copy-mib", type=int, default=0,
                    help="after timing, copy this many MiB device-to-device once (a plain copy "
                         "of known size that scales the FETCH_SIZE/WRITE_SIZE counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: the render path has no multi-GPU form (asked for "
              f"--gpus {args.gpus})", file=sys.stderr)
        sys.exit(2)

    cu = importlib.import_module("chaos-ultra_amd")
    cu.init(0)
    engine = cu.Engine()
    if args.leg != "all":
        leg = {"c1": lambda: c1_leg(cu, engine)[0],
               "uneven": lambda: uneven_leg(cu, engine), "deep": lambda: deep_leg(cu, engine),
               "serving": lambda: serving_leg(cu), "renderer": lambda: renderer_leg(cu),
               "serving_capacity": lambda: serving_capacity_leg(cu)}[args.leg]()
        calibrate_copy(cu, args.calibrate_copy_mib)
        engine.close()
        print(json.dumps({"leg": args.leg, "result": leg}), flush=True)
        return
    tile = frame_tile(cu)

    log(f"[bench] FP64 frame {W}x{H} spp={SPP} maxIter={MAX_ITER} pipeline tune={TUNE}")
    run = PipelineRun(cu, engine, tile, 64, TUNE)
    dt, iters, iters1 = timed(cu, run, args.steps, args.warmup)
    value = iters * args.steps / dt / 1e9
    ms_step = dt / args.steps * 1e3
    pass1_ms = float(np.mean(run.pass1_ms))
    render_ms = np.array(run.total_ms)
    achieved = iters1 * FLOPS_PER_ITER / (pass1_ms * 1e-3) / 1e12
    frame_tflops = iters * FLOPS_PER_ITER / (float(np.mean(render_ms)) * 1e-3) / 1e12
    log(f"[bench] FP64 {value:.1f} G-iter/s, {ms_step:.3f} ms/step, pass 1 {pass1_ms:.3f} ms "
        f"({iters1 / iters:.3f} of the iterations), render p50 {np.median(render_ms):.3f} ms")
    # end to end (outside the timed steps): a render, then the RGBA8 image copied to
    # ordinary host memory, as a caller reading the frame into its own array would
    host = np.empty(W * H, dtype=np.uint32)
    e2e_ms, copy_ms = [], []
    for _ in range(5):
        t0 = time.perf_counter()
        run.step()
        cu.synchronize()
        t1 = time.perf_counter()
        cu.abi.call("cu_memcpy_dtoh", host.ctypes.data_as(ctypes.c_void_p), run.rgba.ptr,
                    ctypes.c_size_t(host.nbytes))
        t2 = time.perf_counter()
        e2e_ms.append((t2 - t0) * 1e3)
        copy_ms.append((t2 - t1) * 1e3)
    # the same into page-locked host memory (cu_host_alloc)
    pinned = cu.HostBuffer(host.nbytes)
    e2e_pin, copy_pin = [], []
    for _ in range(5):
        t0 = time.perf_counter()
        run.step()
        cu.synchronize()
        t1 = time.perf_counter()
        pinned.download_from(run.rgba)
        t2 = time.perf_counter()
        e2e_pin.append((t2 - t0) * 1e3)
        copy_pin.append((t2 - t1) * 1e3)
    pinned.close()
    frame_counts, frame_smooth = run.frame.counts(), run.frame.smooth()

    def readback_of(e2e, cp):
        return {"frame_ms_p50": round(float(np.median(e2e)), 3),
                "copy_ms_p50": round(float(np.median(cp)), 3),
                "copy_gb_s": round(host.nbytes / (float(np.median(cp)) * 1e-3) / 1e9, 1),
                "giga_iter_s": round(iters / (float(np.median(e2e)) * 1e-3) / 1e9, 1)}
    readback = {"pageable": readback_of(e2e_ms, copy_ms), "page_locked": readback_of(e2e_pin, copy_pin),
                "note": "render + device-to-host copy of the 64 MiB RGBA8 image into ordinary "
                        "(pageable) or cu_host_alloc (page-locked) host memory; not part of value "
                        "(the image stays in HBM)"}
    log(f"[bench] with read-back: {readback}")
    run.close()

    variants = {}
    c1_planes = None
    if not args.no_variants:
        log("[bench] C1 frame (1024x1024, maxIter 1000)")
        variants["c1_plain_1024"], c1_planes = c1_leg(cu, engine)
        log(f"[bench] C1: {variants['c1_plain_1024']}")
        vsteps = max(3, args.steps // 2)
        g = GridRun(cu, engine, tile, 64)
        dt2, it2, _ = timed(cu, g, vsteps, 1)
        variants["fp64_grid_kernel"] = {"giga_iter_s": round(it2 * vsteps / dt2 / 1e9, 1),
                                        "kernel_ms": round(float(np.mean(g.pass1_ms)), 3)}
        log(f"[bench] FP64 grid kernel: {variants['fp64_grid_kernel']}")
        r32 = PipelineRun(cu, engine, tile, 32, TUNE)
        dt3, it3, _ = timed(cu, r32, vsteps, 1)
        variants["fp32_pipeline"] = {
            "giga_iter_s": round(it3 * vsteps / dt3 / 1e9, 1),
            "render_ms_p50": round(float(np.median(r32.total_ms)), 3),
            "note": "FP32 c-grid at this zoom is coarser than the pixel (pixel 2.4e-8 < "
                    "ulp_f32(0.74) 5.96e-8): a throughput figure, not an image"}
        log(f"[bench] FP32 pipeline: {variants['fp32_pipeline']}")
        r32.close()
        log("[bench] uneven tiles (256, autotuned)")
        variants["uneven_tiles_256"] = uneven_leg(cu, engine)
        u = variants["uneven_tiles_256"]
        log(f"[bench] uneven tiles: pipeline {u['tuned_pipeline']}, winner {u['autotune']['engine']} "
            f"{u.get('tuned_persistent', u['tuned_pipeline'])}")
        log("[bench] serving: 16 zoom sessions in real time")
        variants["serving_16_sessions"] = serving_leg(cu)
        log(f"[bench] serving: {variants['serving_16_sessions']}")
        log("[bench] serving capacity: 4K sessions at 30 fps within a 33 ms p99")
        variants["serving_capacity_4k"] = serving_capacity_leg(cu)
        variants["renderer_4k"] = renderer_leg(cu)
        log(f"[bench] renderer (drop-in path) 3840x2160: {variants['renderer_4k']}")
        log("[bench] deep zoom 1920x1080")
        variants["deep_zoom_1080p"] = deep_leg(cu, engine)
        variants["iterations_note"] = COUNTED
        log(f"[bench] deep zoom: {json.dumps(variants['deep_zoom_1080p'])}")

    result = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "Giga-iter/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_step, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "plain Mandelbrot FP64 4096x4096, 4 jittered spp (SplitMix64 seed "
                               f"{SEED}), centre (-0.743643887037151, 0.131825904205330), width 1e-4, "
                               "maxIter 5000, bailout |z|^2>=256, smooth value + RGBA8 compose "
                               "(256-entry palette)",
                   "kernel": "frame pipeline (pass 1 + the persistent drain of its straggler queue + combine)",
                   "tune": {"block_steps": TUNE[0], "handoff_lanes": TUNE[1],
                            "tail_passes": TUNE[2], "drain_refill": TUNE[3]},
                   "iterations_per_step": int(iters),
                   "iterations_note": "iterations of the reference's loop, 99.5 % of them run: interior "
                                      "orbits found to be cycles stop early",
                   "render_ms_p50": round(float(np.median(render_ms)), 3),
                   "render_ms_p99": round(float(np.percentile(render_ms, 99)), 3),
                   "with_readback": readback},
        "roofline": {"bound": "valu", "achieved": round(achieved, 2), "peak": FP64_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": round(achieved / FP64_PEAK_TFLOPS, 4),
                     "traffic": read_traffic(),
                     "kernel": "escapePass1DoubleFusedK%d" % TUNE[0],
                     "kernel_ms": round(pass1_ms, 4),
                     "iterations_per_launch": int(iters1),
                     "flops_per_iteration": FLOPS_PER_ITER,
                     "issue_ceiling_giga_iter_s": round(FP64_ISSUE_CEILING_GITER, 1),
                     "frac_of_issue_ceiling": round(iters1 / (pass1_ms * 1e-3) / 1e9
                                                    / FP64_ISSUE_CEILING_GITER, 4),
                     "whole_frame_tflops": round(frame_tflops, 2)},
        "variants": variants,
    }
    if not args.no_cpu:
        log("[bench] CPU baseline (oracle, bounded sample)")
        result["cpu_baseline"] = cpu_baseline(cu, tile, frame_counts, frame_smooth, c1_planes)
        log(f"[bench] CPU {result['cpu_baseline']['value']} G-iter/s, band vs GPU frame "
            f"{result['cpu_baseline'].get('vs_gpu_frame')}")
    calibrate_copy(cu, args.calibrate_copy_mib)
    engine.close()
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
