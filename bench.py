#!/usr/bin/env python3
"""Benchmark: split-steps/s of the fused 2-D split step at 2048^2 complex64.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--local]

A step is one split step (linear step in Fourier space + real-space
nonlinear step) of the 2048x2048 complex64 field of the speckle workload:
alpha=20, n2=-1.6e-9, Isat=1e5, real potential V, dz=5e-6, speckle input,
and the nonlocal response of nl_length = 20 um (the reference's K0 kernel:
d = nl_length // dX = 4 points, a 25x25 kernel applied as a zero-padded
linear convolution), with the field resident in HBM.  ``--local`` drops the
nonlocal term (two sweeps per step).

Printed: one JSON line with the throughput, the roofline of the dominant
kernel (its average duration measured with HIP events on the engine's
stream), the per-kernel and step-level byte counts, and the CPU baseline
(the oracle's complex64 path on the host cores, a bounded sample of the
same workload).
"""

from __future__ import annotations

import argparse
import json
import os
import platform
import sys
import time

import numpy as np

HBM_PEAK = 8.0e12  # MI355X HBM3E, B/s
PROFILES = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles")
PROFILE = {False: os.path.join(PROFILES, "split_step_nonlocal_2048_c64.md"),
           True: os.path.join(PROFILES, "split_step_2048_c64.md")}


def measured_traffic(sweep: str, grid: int, local: bool):
    """HBM bytes per launch of a kernel from the committed rocprofv3
    FETCH_SIZE/WRITE_SIZE summary (2048^2 workloads only), else None."""
    path = PROFILE[local]
    if grid != 2048 or not os.path.exists(path):
        return None
    try:
        text = open(path).read()
        block = text.split("```json", 1)[1].split("```", 1)[0]
        return float(json.loads(block)[sweep]["traffic_bytes"])
    except (IndexError, KeyError, ValueError):
        return None


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def cpu_baseline(N: int, budget_s: float, threads: int, nl_length: float, mode: str = "k0") -> dict:
    """Oracle (complex64, scipy single-precision FFT, elementwise steps on a
    thread pool, scipy oaconvolve for the nonlocal term) on the host cores:
    steps of the same 2048^2 workload until `budget_s` of wall time has
    passed."""
    import oracle
    from nlse_amd import workloads as W

    sim = W.speckle_nonlocal_nlse(oracle.NLSE, N, nonlocal_length=nl_length, fft="pocketfft32", workers=threads,
                    threads=threads)
    sim.nonlocal_mode = mode
    E0 = W.speckle_field(sim)
    A, A_sq = sim._prepare_output_array(E0, True)
    prop = sim._build_propagator()
    V = np.array(sim.V, copy=True)
    sim.split_step(A, A_sq, V, prop, "single")  # warm-up (planning, pools)
    n, t0 = 0, time.perf_counter()
    while True:
        sim.split_step(A, A_sq, V, prop, "single")
        n += 1
        el = time.perf_counter() - t0
        if el >= budget_s and n >= 2:
            break
    return {
        "value": n / el,
        "unit": "split-steps/s",
        "cores": threads,
        "kind": "port",
        "sample": f"{n} split steps of the {N}x{N} speckle workload "
                  f"({('nonlocal, ' + ('FP64 FFT Lorentzian' if mode == 'lorentzian' else 'scipy oaconvolve')) if nl_length > 0 else 'without the nonlocal term'}) on the "
                  f"CPU oracle: complex64, scipy.fft single precision with {threads} workers, elementwise "
                  f"steps on {threads} threads; {el:.1f} s; host CPU: {cpu_model()} "
                  f"(os.cpu_count()={os.cpu_count()})",
    }


def kernel_bytes(P: int, N: int, r: int, local: bool, lorentzian: bool = False) -> dict:
    """Algorithmic HBM bytes per launch of each kernel of the step (P field
    points, complex64 field, float32 V).  Nonlocal one-component fields use
    the packed intensity torus of P/2 complex points (4 B per field point)
    and band points within r of its edges; the Fourier-space (Lorentzian)
    response packs rows the same way and has no band points."""
    if local:
        return {"row": (0, P * (16 + 4)), "col": (1, P * 16)}
    if lorentzian:
        # row pairs packed into one complex intensity line (4 B per field
        # point), the full-torus spectrum quadrant
        khat = 4 * (N // 2 + 1) * (N // 2 + 1)
        return {
            "col": (1, P * 16),
            "nlc_z": (2, P * (8 + 8 + 4)),
            "colZ": (4, P * 8 + khat),
            "nlc_nl": (5, P * (8 + 4 + 4 + 8)),
        }
    band = 4 * r * N + (N - 4 * r) * 2 * r
    khat = 4 * (N // 4 + 1) * (N // 2 + 1)
    return {
        "col": (1, P * 16),                               # field F_y, P, I_y
        "nlc_z": (2, P * (8 + 8 + 4)),                    # field in/out, Z out
        "band": (3, band * (8 + 4)),                      # field at band points, values out
        "colZ": (4, P * 8 + khat),                        # Z in/out, kernel spectrum
        "nlc_nl": (5, P * (8 + 4 + 4 + 8) + band * 4),    # field, Z, V in; field out
        "band+colZ": (6, band * (8 + 4) + P * 8 + khat),  # the two above in one launch (as the step runs them)
    }


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--workload", choices=("speckle", "batch", "gvd3d", "corrector"), default="speckle",
                    help="speckle: 2048^2 nonlocal split step (the metric); batch: 64 uneven fields; "
                         "gvd3d: 3-D 512x512x64 with GVD; corrector: learned corrector at 1024^2")
    ap.add_argument("--steps", type=int, default=None)
    ap.add_argument("--warmup", type=int, default=None)
    ap.add_argument("--grid", type=int, default=2048)
    ap.add_argument("--local", action="store_true", help="drop the nonlocal term (speckle-workload physics otherwise)")
    ap.add_argument("--nonlocal-mode", choices=("k0", "lorentzian"), default="k0",
                    help="k0: the reference's K0 convolution; lorentzian: 1/(1+(k l)^2) in Fourier space")
    ap.add_argument("--col-width", type=int, default=0, help="columns per block of the column sweep (0: default)")
    ap.add_argument("--row-points", type=int, default=0,
                    help="points per thread of the x-row kernels, i.e. their radix plan (0: default, 8 or 16)")
    ap.add_argument("--graph-chunk", type=int, default=-1,
                    help="steps per captured graph launch (-1: the engine's default, 0: no graph)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-e2e", action="store_true", help="skip the end-to-end out_field timings")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--width", type=int, default=32, help="corrector: channels of the network")
    ap.add_argument("--pairs", type=int, default=20000, help="corrector: streamed training pairs")
    ap.add_argument("--eval-seeds", type=int, default=200, help="corrector: held-out seeds")
    ap.add_argument("--no-corrector", action="store_true", help="skip the corrector summary of the default line")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported (the engine runs one process "
              "on one GPU; sharding across GPUs is not built).", file=sys.stderr)
        return 2
    defaults = {"speckle": (1000, 50), "batch": (500, 20), "gvd3d": (200, 10), "corrector": (100, 5)}[args.workload]
    args.steps = defaults[0] if args.steps is None else args.steps
    args.warmup = defaults[1] if args.warmup is None else args.warmup
    if args.workload == "batch":
        return bench_batch(args)
    if args.workload == "gvd3d":
        return bench_gvd3d(args)
    if args.workload == "corrector":
        return bench_corrector(args)
    return bench_speckle(args)


def bench_speckle(args) -> int:
    import torch

    from nlse_amd import NLSE
    from nlse_amd import workloads as W

    N = args.grid
    nl_length = 0.0 if args.local else 20e-6
    sim = W.speckle_nonlocal_nlse(NLSE, N, nonlocal_length=nl_length)
    sim.col_width = args.col_width
    sim.row_points = args.row_points
    lorentzian = not args.local and args.nonlocal_mode == "lorentzian"
    if lorentzian:
        sim.nonlocal_mode = "lorentzian"
    E0 = W.speckle_field(sim)
    sim._own_propagator()
    sim._send_arrays_to_gpu()
    A, _ = sim._prepare_output_array(E0, True)
    eng = sim._engine_for(A)
    if args.graph_chunk >= 0:
        eng.graph_chunk = args.graph_chunk
    sim._configure(eng, A, sim.V, sim.propagator, "single")
    P = A.numel()
    r = 0 if args.local else int(tuple(sim.nl_profile.shape)[0] // 2)
    kb = kernel_bytes(P, N, r, args.local, lorentzian)
    # one step's launches: the shared band+colZ entry repeats the bytes of
    # the band and colZ entries (timed alone for reference)
    step_bytes = sum(b for name, (_, b) in kb.items() if name != "band+colZ")

    # warm-up, graph capture (no steps run), then K steps bracketed by
    # synchronisation: the timed region replays an already uploaded graph
    eng.run(A, args.warmup)
    eng.prepare_graph(A)
    torch.cuda.synchronize()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record()
    eng.run(A, args.steps)
    ev1.record()
    torch.cuda.synchronize()
    t_steps = ev0.elapsed_time(ev1) * 1e-3
    steps_per_s = args.steps / t_steps
    finite = bool(torch.isfinite(torch.view_as_real(A)).all())

    # each kernel alone, same stream, same launch configuration
    scratch = A.clone()
    if not args.local:
        eng.run(scratch, 1)  # fills the intensity and band buffers
    kern = {}
    for name, (which, nbytes) in kb.items():
        eng.run_pass(scratch, which, 10)
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        eng.run_pass(scratch, which, args.steps)
        e1.record()
        torch.cuda.synchronize()
        avg = e0.elapsed_time(e1) * 1e-3 / args.steps
        kern[name] = {"avg_us": avg * 1e6, "bytes": nbytes, "GBps": nbytes / avg / 1e9}
    dom = max(kern, key=lambda k: kern[k]["avg_us"])
    achieved = kern[dom]["bytes"] / (kern[dom]["avg_us"] * 1e-6)
    row_points, col_width = eng.config()

    physics = ("real float32 potential, Isat=1e5, alpha=20, dz=5e-6, speckle input (seed 1), "
               "precision='single'")
    if args.local:
        workload = f"speckle-workload physics without the nonlocal term: {N}x{N} complex64 NLSE split step, " + physics
    elif lorentzian:
        workload = (f"{N}x{N} complex64 NLSE split step with the nonlocal response applied in "
                    "Fourier space as 1/(1+(k l)^2), l = 20 um (periodic), " + physics)
    else:
        workload = (f"{N}x{N} complex64 NLSE split step with the nonlocal response "
                    f"(nl_length 20 um, reference K0 kernel {2 * r + 1}x{2 * r + 1}, zero-padded linear "
                    "convolution), " + physics)
    result = {
        "metric": "split-steps/s at 2048^2 c64",
        "value": steps_per_s,
        "unit": "split-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t_steps / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64",
        "data": "synthetic",
        "config": {
            "workload": workload,
            "grid": [N, N],
            "nonlocal_kernel": None if args.local else ("lorentzian" if lorentzian else [2 * r + 1, 2 * r + 1]),
            "kernels": {"row_points_per_thread": row_points, "col_width": col_width},
        },
        "roofline": {
            "bound": "hbm",
            "kernel": dom,
            "achieved": achieved / 1e9,
            "peak": HBM_PEAK / 1e9,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK,
            "traffic": None if lorentzian else measured_traffic(dom, N, args.local),
        },
        "kernels": kern,
        "step_roofline": {
            "bytes_per_step": step_bytes,
            "B_per_point": step_bytes / P,
            "achieved_GBps": steps_per_s * step_bytes / 1e9,
            "frac": steps_per_s * step_bytes / HBM_PEAK,
            "min_B_per_point": 36 if args.local else 52,
            "frac_of_min_schedule": steps_per_s * P * (36 if args.local else 52) / HBM_PEAK,
        },
        "grid_point_steps_per_s": steps_per_s * P,
        "field_finite": finite,
    }
    if not args.no_e2e:
        result["end_to_end"] = end_to_end(N, nl_length, lorentzian)
    if not lorentzian:
        result["complex128"] = complex128_summary(N, nl_length, min(args.steps, 50))
    if not args.no_corrector and not args.local:
        result["corrector"] = corrector_summary(args)
    if not args.no_cpu:
        threads = min(os.cpu_count() or 1, 16)
        result["cpu_baseline"] = cpu_baseline(N, args.cpu_seconds, threads, nl_length,
                                              "lorentzian" if lorentzian else "k0")
    print(json.dumps(result), flush=True)
    return 0


def complex128_summary(N: int, nl_length: float, steps: int) -> dict:
    """The same workload with a complex128 field (propagated in FP64 by the
    complex128 kernels, as the reference keeps E_in's precision): steady
    split steps per second with the field resident, graph replay as above."""
    import torch

    from nlse_amd import NLSE
    from nlse_amd import workloads as W

    sim = W.speckle_nonlocal_nlse(NLSE, N, nonlocal_length=nl_length)
    E0 = W.speckle_field(sim).astype(np.complex128)
    sim._own_propagator()
    sim._send_arrays_to_gpu()
    A, _ = sim._prepare_output_array(E0, True)
    eng = sim._engine_for(A)
    sim._configure(eng, A, sim.V, sim.propagator, "single")
    eng.run(A, 3)
    eng.prepare_graph(A)
    torch.cuda.synchronize()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record()
    eng.run(A, steps)
    ev1.record()
    torch.cuda.synchronize()
    t = ev0.elapsed_time(ev1) * 1e-3
    sim._retrieve_arrays_from_gpu()
    return {"split_steps_per_s": steps / t, "ms_per_step": t / steps * 1e3, "steps": steps,
            "grid_point_steps_per_s": steps / t * A.numel(), "dtype": "c128 (FP64 storage and arithmetic)",
            "field_finite": bool(torch.isfinite(torch.view_as_real(A)).all())}


def end_to_end(N: int, nl_length: float, lorentzian: bool) -> dict:
    """Wall time of whole out_field calls, host (numpy) field in and out, the
    way the reference's published figure times them (propagator, plans,
    transfers and normalisation included): the speckle-workload run over its full
    length, and the settings of the reference's own 2-D benchmark
    (examples/fig1_benchmarks.py: L = 2 mm, dz = 1e-4, 20 steps, V = None,
    alpha = 22, Isat = 3.92e4, n2 = -1.99e-9, P = 1.05 W, window 11.3 mm,
    mean of two calls on one instance),
    which the reference reports at about 0.38 s at 2048^2 on an RTX 4090."""
    import torch

    from nlse_amd import NLSE
    from nlse_amd import workloads as W
    from nlse_amd.nlse import count_steps

    sim = W.speckle_nonlocal_nlse(NLSE, N, nonlocal_length=nl_length)
    if lorentzian:
        sim.nonlocal_mode = "lorentzian"
    E0 = W.speckle_field(sim)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    out = sim.out_field(E0, sim.L, verbose=False)
    t_full = time.perf_counter() - t0
    n_full = count_steps(sim.L, sim.delta_z)
    # examples/fig1_benchmarks.py:17-59: window 3008 x 3.76 um, waist 2.29 mm,
    # I_sat set after construction, the propagator built by the first call
    ref = NLSE(alpha=22, power=1.05, window=3008 * 3.76e-6, n2=-1.99e-9, V=None, L=2e-3, NX=N, NY=N)
    ref.I_sat = 3.92e4
    ref.delta_z = 1e-4
    G = np.exp(-(np.hypot(ref.XX, ref.YY) ** 2) / 2.29e-3**2).astype(np.complex64)
    times = []
    for _ in range(2):
        t0 = time.perf_counter()
        ref.out_field(G, 2e-3, verbose=False)
        times.append(time.perf_counter() - t0)
    return {
        "speckle_nonlocal_full_length": {"seconds": t_full, "steps": n_full, "steps_per_s_incl_overhead": n_full / t_full,
                                "finite": bool(np.isfinite(out).all())},
        "reference_fig1_settings": {"seconds_mean_of_2": float(np.mean(times)), "steps": count_steps(2e-3, 1e-4),
                                    "published_rtx4090_seconds": 0.38 if N == 2048 else None},
    }


def _timed(fn, *a) -> float:
    """Seconds of one call of fn, bracketed by synchronisation and HIP
    events on the current stream."""
    import torch

    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    fn(*a)
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e-3


def bench_batch(args) -> int:
    """Uneven batch: 64 fields of 256^2/512^2/1024^2 with random n2, power,
    Isat, one launch per sweep and line length for the whole batch (or one per
    sweep), steady steps replayed from a captured graph.  Compared with the
    same fields run one after the other through their own plans."""
    import torch

    from nlse_amd import NLSE, NLSEBatch
    from nlse_amd import workloads as W

    sims, fields = W.uneven_batch(NLSE)
    batch = NLSEBatch(sims)
    eng, buf, _ = batch.prepare(fields, 1e-5)
    P = eng.total
    # both launch structures: one persistent launch per sweep for all line
    # lengths, and one per length present; the line reports the faster
    modes = {}
    for single in (True, False):
        eng.set_single_launch(single)
        eng.run(buf, args.warmup)
        eng.prepare_graph(buf)
        modes["single_launch" if single else "per_length_launches"] = _timed(eng.run, buf, args.steps)
    best = min(modes, key=modes.get)
    eng.set_single_launch(best == "single_launch")
    t = modes[best]
    sps = args.steps / t
    finite = bool(torch.isfinite(torch.view_as_real(buf)).all())
    kern = {}
    for name, which, nbytes in (("row", 0, P * 16), ("col", 1, P * 16)):
        eng.run_pass(buf, which, 5)
        avg = _timed(eng.run_pass, buf, which, args.steps) / args.steps
        kern[name] = {"avg_us": avg * 1e6, "bytes": nbytes, "GBps": nbytes / avg / 1e9}
    dom = max(kern, key=lambda k: kern[k]["avg_us"])
    achieved = kern[dom]["bytes"] / (kern[dom]["avg_us"] * 1e-6)
    # the same fields through separate plans, one after the other
    seq = []
    for s, E in zip(sims, fields):
        s._own_propagator()
        s._send_arrays_to_gpu()
        A, _ = s._prepare_output_array(E, True)
        e = s._engine_for(A)
        s._configure(e, A, s.V, s.propagator, "single")
        seq.append((e, A))
    nseq = max(10, args.steps // 10)
    for e, A in seq:
        e.run(A, 2)
    t_seq = _timed(lambda: [e.run(A, nseq) for e, A in seq]) / nseq
    result = {
        "metric": "batch split-steps/s (64 uneven fields, every field one step)",
        "value": sps,
        "unit": "batch-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64",
        "data": "synthetic",
        "config": {"workload": "64 NLSE fields, N uniform on {256, 512, 1024} (rng 2), n2 = -10^U(-10,-8), "
                               "P ~ U(0.1, 2) W, Isat ~ U(1e4, 1e6), alpha=20, V=None, dz=1e-5, precision='single'",
                   "points": P, "batch": eng.config(), "graph_chunk": eng.graph_chunk, "launches": best,
                   "ms_per_step_by_launch_structure": {k: v / args.steps * 1e3 for k, v in modes.items()}},
        "roofline": {"bound": "hbm", "kernel": f"batch {dom} sweep", "achieved": achieved / 1e9,
                     "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": achieved / HBM_PEAK, "traffic": None},
        "kernels": kern,
        "step_roofline": {"B_per_point": 32, "achieved_GBps": sps * P * 32 / 1e9, "frac": sps * P * 32 / HBM_PEAK},
        "grid_point_steps_per_s": sps * P,
        "separate_plans_steps_per_s": 1.0 / t_seq,
        "batch_speedup_vs_separate": sps * t_seq,
        "field_finite": finite,
    }
    if not args.no_cpu:
        import oracle

        threads = min(os.cpu_count() or 1, 16)
        osims, ofields = W.uneven_batch(oracle.NLSE, fft="pocketfft32", workers=threads, threads=threads)
        t0, n, pts = time.perf_counter(), 0, 0
        for s, E in zip(osims, ofields):
            A, A_sq = s._prepare_output_array(E, True)
            prop = s._build_propagator()
            s.split_step(A, A_sq, None, prop, "single")
            n += 1
            pts += E.size
            if time.perf_counter() - t0 > args.cpu_seconds:
                break
        el = time.perf_counter() - t0
        result["cpu_baseline"] = {
            "value": pts / el / P, "unit": "batch-steps/s", "cores": threads, "kind": "port",
            "sample": f"one split step of each of the first {n} batch fields on the CPU oracle (complex64, "
                      f"scipy.fft with {threads} workers), {pts} grid points in {el:.1f} s, scaled to the batch's "
                      f"{P} points; host CPU: {cpu_model()}"}
    print(json.dumps(result), flush=True)
    return 0


def bench_gvd3d(args) -> int:
    """3-D (x, y, t) NLSE 512x512x64 with GVD: four sweeps per step."""
    import torch

    from nlse_amd import NLSE_3d
    from nlse_amd import workloads as W

    sim = W.gvd_3d(NLSE_3d)
    E0 = W.sech_pulse_field(sim)
    sim._own_propagator()
    sim._send_arrays_to_gpu()
    A, _ = sim._prepare_output_array(E0, True)
    eng = sim._engine_for(A)
    sim._configure(eng, A, sim.V, sim.propagator, "single")
    P = A.numel()
    cell = sim.delta_X * sim.delta_Y * sim.delta_T

    def energy():
        return float(torch.view_as_real(A).double().pow(2).sum()) * cell * 299792458.0 * 8.8541878128e-12 / 2

    e_start = energy()
    eng.run(A, args.warmup)
    eng.prepare_graph(A)
    t = _timed(eng.run, A, args.steps)
    e_end = energy()
    sps = args.steps / t
    nbytes = P * 64  # four sweeps of 16 B/pt (V = None)
    result = {
        "metric": "split-steps/s, 3-D NLSE 512x512x64 c64",
        "value": sps,
        "unit": "split-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64",
        "data": "synthetic",
        "config": {"workload": "NLSE_3d 512x512x64, D0=-1e-26, window [4e-3, 4e-3, 2e-12], n2=-1e-9, "
                               "alpha=0, Isat=inf, dz=1e-5, Gaussian x sech(t/200fs), precision='single'",
                   "grid": list(A.shape)},
        "roofline": {"bound": "hbm", "kernel": "step (4 sweeps)", "achieved": sps * nbytes / 1e9,
                     "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": sps * nbytes / HBM_PEAK, "traffic": None},
        "step_roofline": {"B_per_point": 64, "min_B_per_point": 48, "frac_of_min_schedule": sps * P * 48 / HBM_PEAK},
        "grid_point_steps_per_s": sps * P,
        "energy_drift_per_step": (e_end - e_start) / e_start / (args.warmup + args.steps),
    }
    print(json.dumps(result), flush=True)
    return 0


def corrector_summary(args, N: int = 1024, seeds=(301, 302, 303, 304)) -> dict:
    """Learned corrector, short form for the default line: a network trained
    at 128^2 (1600 pairs from the plain solver, 800 Adam steps on the GPU)
    applied at N^2 with the same weights (the spectral weights act on the
    same 32 x 32 physical modes), against plain settings at equal error over
    L = 10 mm on a few held-out seeds (corrector.equal_error_study); the
    full-size study is --workload corrector."""
    import torch

    from nlse_amd import corrector as CR
    from nlse_amd.fno import FNO

    t0 = time.perf_counter()
    pairs = CR.make_pairs(N=128, trajectories=80, coarse_steps=20, seed=1)
    net = FNO(128, 128, width=args.width, layers=4, seed=0)
    CR.train(net, pairs, steps=800, batch=8, lr=2e-3)
    torch.cuda.synchronize()
    t_train = time.perf_counter() - t0
    del pairs
    big = FNO(N, N, width=args.width, layers=4, params=net.params())
    big.res_scale = net.res_scale
    st = CR.equal_error_study(big, N, seeds)
    st["train"] = {"grid": 128, "pairs": 1600, "adam_steps": 800, "seconds": t_train}
    st["reference"] = "plain fine-step solution (Lie, dz = 1e-5) on the GPU, the solver the corrector reproduces"
    return st


def bench_corrector(args) -> int:
    """Learned corrector at its configuration: 2-D NLSE at 1024^2, FNO of 4
    spectral layers, 32 channels, 32 x 32 modes, BF16 MFMA; coarse steps of
    8e-5 corrected towards 8 fine steps of 1e-5.  Training on a stream of
    20k (coarse, fine) pairs made on the fly by the plain solver (README
    material x U(0.5, 1.5), speckle inputs); evaluation on 200 held-out seeds
    over L = 10 mm against the fine-step solution, with the power/Hamiltonian
    fallback; throughput compared with the fine steps and with the fastest
    plain setting (Lie or Strang, larger dz) of equal error.  One seed is
    also checked against the FP64 oracle of the fine-step scheme."""
    import numpy as np
    import torch

    import oracle
    from nlse_amd import corrector as CR
    from nlse_amd.fno import FNO

    N = args.grid if args.grid != 2048 else 1024
    pairs = args.pairs
    seeds = list(range(10_000, 10_000 + args.eval_seeds))
    net = FNO(N, N, width=args.width, layers=4, seed=0)
    t0 = time.perf_counter()
    tr = CR.train_stream(net, N, pairs, batch=8, lr=2e-3, seed=1, log_every=250)
    torch.cuda.synchronize()
    t_train = time.perf_counter() - t0
    print(f"[corrector] trained on {tr['pairs']} streamed pairs at {N}^2 in {t_train:.0f} s", flush=True)
    st = CR.equal_error_study(net, N, seeds, log_every=20)
    print(f"[corrector] {len(seeds)} held-out seeds evaluated", flush=True)
    diag = CR.rollout_diagnostics(net, N, seeds[:20])
    print(f"[corrector] single-step and damped-rollout diagnostics done", flush=True)
    # the reference itself against the FP64 oracle of the fine-step scheme
    rng = np.random.default_rng(seeds[0])
    mat = CR.material(rng)
    kw = dict(alpha=mat["alpha"], power=mat["power"], window=CR.WINDOW, n2=mat["n2"], V=None, L=10e-3, NX=N, NY=N,
              Isat=mat["Isat"])
    from nlse_amd import NLSE

    E0 = CR._speckle_field(NLSE(**kw), rng)
    ref, _ = CR._propagate(N, mat, E0, 1e-5, 10e-3)
    o = oracle.NLSE(mode="c128", workers=min(os.cpu_count() or 1, 16), threads=min(os.cpu_count() or 1, 16), **kw)
    o.delta_z = 1e-5
    r128 = o.out_field(E0.astype(np.complex128), 10e-3 - 0.5e-5)  # 1000 steps, as the reference run
    fine_vs_fp64 = float(np.linalg.norm(ref.cpu().numpy() - r128) / np.linalg.norm(r128))
    x_in = torch.zeros(1, 4, N, N, device="cuda")
    net.forward(x_in)
    t_net = _timed(net.forward, x_in)
    result = {
        "metric": "corrector vs plain at equal relative L2 error (1024^2 c64)",
        "value": st["speedup_vs_equal_error_plain"],
        "unit": "x (time of the equal-error plain setting / time of the corrected loop)",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": st["corrected"]["seconds"] / max(1, st["corrected"]["coarse_steps"] // len(seeds)) * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64 solver, bf16 MFMA network (fp32 accumulation)",
        "data": "synthetic",
        "config": {"workload": f"FNO corrector (4 spectral layers, {args.width} channels, 32x32 modes) of coarse "
                               f"steps dz_c = 8e-5 vs 8 fine steps of 1e-5 at {N}^2; trained on {tr['pairs']} "
                               "pairs streamed from the plain solver (README material x U(0.5,1.5), speckle "
                               f"inputs); evaluated on {len(seeds)} held-out seeds over L = 10 mm",
                   "train_seconds": t_train, "train": tr},
        "study": st,
        "rollout_diagnostics": diag,
        "speedup_vs_fine": st["speedup_vs_fine"],
        "network_ms": t_net * 1e3,
        "fine_reference_vs_fp64_oracle": fine_vs_fp64,
    }
    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
