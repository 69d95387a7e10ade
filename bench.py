#!/usr/bin/env python3
"""SRM throughput on one MI355X: point-harmonics per second.

A step is one SRM realization on the device with its harmonic table already
resident in HBM: per-axis operand tables, the field kernel, the FP64
statistics pass and the rescale/taper epilogue (scarf_srm_run). Host
sampling of the harmonics (the reference's draw loop) is timed separately,
and the reference's own call, scarf_execute (draw, device, field returned in
the caller's host array), is timed end to end: the first call of the process
and warm calls, with the draw streamed into the device work and without.
The 64-realization ensemble runs after it, in the same process.

Default workload (the configuration the metric is quoted on): structured
512 x 512 x 512 grid, dh = 20 m, von Karman Hurst 0.1, cl = 5000 m,
sigma = 0.05, 20000 harmonics, seed 1234. The primary value is the split-bf16
(3-term, 6-product) MFMA kernel; the FP32 direct-sum kernel is measured on
the same resident table for the speed-up, and every kernel's error is
measured over the whole field against the FP64 kernel, itself checked
against the FP64 CPU oracle at sampled points.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload NAME]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))
sys.path.insert(0, str(ROOT / "tests"))

from scarf3d_amd.workloads import WORKLOADS, ensemble_members, init_library, structured_cfg, workload_cfg  # noqa: E402

METRIC = "SRM Gpt·harm/s at 512³×20k: split-BF16 MFMA vs FP32 direct, err≤1e-5σ"
PEAK_MFMA_TFLOPS = 2500.0  # MI355X dense bf16 / fp16
PEAK_VALU_TFLOPS = 157.3   # MI355X FP32 vector
PEAK_VALU_F64_TFLOPS = 78.6  # MI355X FP64 vector
PEAK_HBM_GBS = 8000.0      # MI355X HBM3E
MFMA_PRODUCTS = {"mfma_bf16x3": 6, "mfma_f16x2": 3, "mfma_bf16x2": 3}

KERNELS = ("mfma_bf16x3", "mfma_f16x2", "mfma_bf16x2", "direct_f32", "direct_f64")
# HBM bytes per launch of the timed kernel, measured with rocprofv3 FETCH_SIZE /
# WRITE_SIZE passes scaled by a 1 GiB device copy (the counters cannot be read
# inside the timed run): 1.038e10 - 1.044e10 B on each of the x-128 tiles the
# tuner picks from (32x8, 64x4, 128x2, 256x1 columns), the mean reported:
# (workload, kernel) -> (bytes, summary file)
TRAFFIC = {
    ("precision_512", "mfma_bf16x3"): (1.041e10, "profiles/mfma_grid_bf16x3_512cube_20k_traffic.md"),
}


def _sig(v, digits=4):
    """v rounded to `digits` significant digits (errors of 1e-6 stay visible)."""
    return float(f"{v:.{digits}g}")


def measure_ensemble(kernel, steps, warmup):
    """The 64-member ensemble: first run (draws, tile rates, graph capture)
    and the device time of warm runs (the graph replay, HIP events)."""
    import scarf3d_amd
    from scarf3d_amd.hip import Hip

    lib = scarf3d_amd.load("f")
    hip = Hip()
    members = ensemble_members()
    work = float(sum(np.prod(m["fe"]) * m["nharm"] for m in members))
    bufs = [hip.empty(int(np.prod(m["fe"])), np.float32) for m in members]
    ptrs = [b.ptr for b in bufs]
    t0 = time.perf_counter()
    log(f"[bench] ensemble of {len(members)}: first run (draws, tile rates, graph capture, run)")
    stats = lib.ensemble_execute(members, ptrs, kernel)
    first_s = time.perf_counter() - t0
    log(f"[bench] ensemble first run {first_s:.2f} s")
    for _ in range(max(0, warmup - 1)):
        lib.ensemble_execute(members, ptrs, kernel)
    dev_ms, wall = [], []
    for _ in range(steps):
        t1 = time.perf_counter()
        stats = lib.ensemble_execute(members, ptrs, kernel)
        wall.append(time.perf_counter() - t1)
        dev_ms.append(lib.ensemble_ms())
    for b in bufs:
        b.free()
    ms = float(np.mean(dev_ms))
    P = MFMA_PRODUCTS[kernel]
    achieved = work * 4 * P / (ms * 1e-3) / 1e12
    log(f"[bench] ensemble: {ms:.3f} ms device, {float(np.mean(wall)) * 1e3:.1f} ms per call")
    return dict(work=work, ms=ms, wall_ms=float(np.mean(wall)) * 1e3, first_s=first_s, achieved=achieved,
                frac=achieved / PEAK_MFMA_TFLOPS, host_s_member=float(np.mean(stats[:, 4].astype(np.float64))),
                members=len(members))


def bench_ensemble(args):
    e = measure_ensemble(args.kernel, args.steps, args.warmup)
    work, ms, achieved = e["work"], e["ms"], e["achieved"]
    out = {
        "metric": "SRM ensemble Gpt·harm/s: 64 uneven realizations, one persistent grouped-GEMM launch in a hipGraph",
        "value": round(work / (ms * 1e-3) / 1e9, 2), "unit": "Gpt·harm/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms, 3), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": args.kernel, "data": "synthetic",
        "config": {"workload": "ensemble_64", "members": e["members"], "point_harmonics": work,
                   "kernel": args.kernel, "host_draw_s_per_step_wall": round(e["wall_ms"] * 1e-3 - ms * 1e-3, 3),
                   "host_draw_s_mean_member": round(e["host_s_member"], 3), "first_run_s": round(e["first_s"], 2)},
        "roofline": {"bound": "mfma", "achieved": round(achieved, 1), "peak": PEAK_MFMA_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(achieved / PEAK_MFMA_TFLOPS, 4), "traffic": None,
                     "kernel": f"mfma_ensemble<{args.kernel}>", "flops_per_point_harmonic": 4 * MFMA_PRODUCTS[args.kernel]},
        "cpu_baseline": None,
    }
    print(json.dumps(out), flush=True)
    return 0


def bench_copy_calibration(args):
    """A device-to-device copy of a known size (1 GiB): the reference point
    that scales rocprofv3's FETCH_SIZE / WRITE_SIZE counters into bytes."""
    from scarf3d_amd.hip import Hip

    import ctypes as C

    hip = Hip()
    n = 1 << 28  # floats
    a = hip.empty(n, np.float32)
    b = hip.empty(n, np.float32)
    a.zero()
    for _ in range(max(1, args.steps)):
        rc = hip.L.hipMemcpy(C.c_void_p(b.ptr), C.c_void_p(a.ptr), C.c_size_t(4 * n), 3)
        assert rc == 0
    hip.synchronize()
    print(json.dumps({"copy_bytes": 4 * n, "copies": max(1, args.steps)}), flush=True)
    a.free()
    b.free()
    return 0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def init(lib, w):
    cfg = workload_cfg(w)
    init_library(lib, cfg)
    return cfg


def time_kernel(lib, hip, kernel, d_field, steps, warmup):
    assert lib.set_kernel(kernel) == 0
    for _ in range(warmup):
        lib.srm_run(d_field.ptr)
    hip.synchronize()
    t0 = time.perf_counter()
    field_ms, total_ms = [], []
    for _ in range(steps):
        stats = lib.srm_run(d_field.ptr)
        t = lib.timings()
        field_ms.append(t["field"])
        total_ms.append(t["total"])
    hip.synchronize()
    wall = (time.perf_counter() - t0) / steps
    return dict(ms_per_step=wall * 1e3, field_ms=float(np.mean(field_ms)), device_ms=float(np.mean(total_ms)),
                stats=stats)


def measure_end_to_end(lib, w, kernel, steps, warmup):
    """The reference's own call end to end on the initialized workload:
    scarf_execute (setup, draw, device work, field copied into the caller's
    host array) and scarf_execute_device (the field left in HBM), wall clock
    per call. The first call of the process also starts the HIP runtime,
    tunes the tile and allocates; warm calls reuse all of that. Each is timed
    with the draw streamed into the device work (the default) and with the
    whole table drawn first (stream_draw = 0)."""
    from scarf3d_amd.hip import Hip

    assert lib.set_kernel(kernel) == 0
    seed = w["seed"]
    host = np.empty(lib.npts, dtype=lib.dtype)
    host.fill(0)  # the caller's field array, its pages already touched
    t0 = time.perf_counter()
    _, st = lib.execute(seed, out=host)
    first_ms = (time.perf_counter() - t0) * 1e3
    if lib.last_error():
        raise RuntimeError(lib.last_error())
    log(f"[bench] first scarf_execute of the process: {first_ms:.1f} ms (host draw {st[4] * 1e3:.1f} ms)")
    hip = Hip()
    d = hip.empty(lib.npts, lib.dtype)

    def timed(call):
        for _ in range(warmup):
            call()
        ms, draw = [], []
        for _ in range(steps):
            t1 = time.perf_counter()
            stats = call()
            ms.append((time.perf_counter() - t1) * 1e3)
            draw.append(float(stats[4]) * 1e3)
        return dict(ms=float(np.mean(ms)), min_ms=float(np.min(ms)), draw_ms=float(np.mean(draw)))

    out = {"first_call_ms": first_ms, "first_call_draw_ms": float(st[4]) * 1e3}
    for mode in (1, 0):
        assert lib.set_option("stream_draw", mode) == 0
        tag = "streamed" if mode else "whole_table"
        out[f"execute_{tag}"] = timed(lambda: lib.execute(seed, out=host)[1])
        out[f"execute_device_{tag}"] = timed(lambda: lib.execute_device(seed, d.ptr))
        log(f"[bench] scarf_execute ({tag}): {out[f'execute_{tag}']['ms']:.1f} ms per call; scarf_execute_device "
            f"{out[f'execute_device_{tag}']['ms']:.1f} ms; host draw {out[f'execute_{tag}']['draw_ms']:.1f} ms")
    assert lib.set_option("stream_draw", 1) == 0
    d.free()
    return out


# FIM at the reference examples' configuration (examples/c/driver.c:76-96,
# :405-430: 500^3, ds = dh = 50 m, von Karman cl = 2000 m, Hurst 0.25,
# sigma 0.05, seed 1235, no padding): internal grid 502^3
FIM_CASE = dict(n=(500, 500, 500), ds=50.0, acf=0, hurst=0.25, cl=(2000.0,) * 3, sigma=0.05, seed=1235)


def fim_bytes(npts, nout):
    """Least HBM bytes of one FIM realization (float library): the half
    spectrum written once and read once (8 B per complex value), the output
    written once (4 B per point). The transform's passes along y and z move
    the half spectrum between them, the last one takes the statistics and
    writes the caller's block, so the fraction of HBM bandwidth this gives is
    a floor."""
    n1, n2, n3 = npts
    half = (n1 // 2 + 1) * n2 * n3
    return 8 * half + 8 * half + 4 * nout


def measure_fim(steps, warmup, cpu=True):
    """FIM (method 0) at FIM_CASE: the first call of the process (runtime,
    transform tables, buffers), then warm scarf_execute_device (field in HBM)
    and scarf_execute (field into a host array) calls, wall clock, with the
    device pass times the library reports in stats(5:8)."""
    import scarf3d_amd
    from scarf3d_amd.hip import Hip

    lib = scarf3d_amd.load("f")
    c = FIM_CASE
    cfg = structured_cfg(n=c["n"], ds=c["ds"], acf=c["acf"], hurst=c["hurst"], cl=c["cl"], sigma=c["sigma"],
                         real=np.float32)
    cfg["method"] = 0
    init_library(lib, cfg)
    hip = Hip()
    d = hip.empty(lib.npts, np.float32)
    t0 = time.perf_counter()
    st = lib.execute_device(c["seed"], d.ptr)
    first_ms = (time.perf_counter() - t0) * 1e3
    if lib.last_error():
        raise RuntimeError(lib.last_error())
    for _ in range(warmup):
        lib.execute_device(c["seed"], d.ptr)
    ms, parts = [], []
    for _ in range(steps):
        t1 = time.perf_counter()
        st = lib.execute_device(c["seed"], d.ptr)
        ms.append((time.perf_counter() - t1) * 1e3)
        parts.append([float(v) * 1e3 for v in st[4:8]])
    host = np.zeros(lib.npts, dtype=np.float32)
    hms = []
    for _ in range(max(2, steps // 2)):
        t1 = time.perf_counter()
        lib.execute(c["seed"], out=host)
        hms.append((time.perf_counter() - t1) * 1e3)
    d.free()
    lib.finalize()
    sys.path.insert(0, str(Path(__file__).resolve().parent / "oracle"))
    import fim_oracle as fo

    s = fo.setup(dict(cfg, pad=0), np.float32)
    npts = s["npts"]
    nint_ = int(np.prod(npts))
    nout = int(np.prod(c["n"]))
    dev = float(np.mean(ms))
    part = np.mean(np.array(parts), axis=0)
    B = fim_bytes(npts, nout)
    out = {"workload": "fim_500", "internal_grid": npts, "first_call_ms": _sig(first_ms), "ms": _sig(dev),
           "min_ms": _sig(float(np.min(ms))), "execute_host_ms": _sig(float(np.mean(hms))),
           "spectrum_ms": _sig(part[0]), "symmetry_ms": _sig(part[1]), "transforms_ms": _sig(part[2]),
           "mapping_ms": _sig(part[3]), "mpts_per_s": _sig(nout / (dev * 1e-3) / 1e6),
           "internal_mpts_per_s": _sig(nint_ / (dev * 1e-3) / 1e6),
           "hbm": {"algorithmic_bytes": B, "achieved_gbs": _sig(B / (dev * 1e-3) / 1e9), "peak_gbs": PEAK_HBM_GBS,
                   "frac": _sig(B / (dev * 1e-3) / 1e9 / PEAK_HBM_GBS)},
           "note": "scarf_execute_device wall clock per call (spectrum, symmetry, dense transform with the "
                   "statistics and the caller's block); stage ms from the library's stats(5:8), HIP events; "
                   "hbm.frac counts the spectrum written and read once and the output written once (fim_bytes)"}
    log(f"[bench] FIM {c['n']} (internal {npts}): first call {first_ms:.1f} ms, {dev:.2f} ms per call "
        f"(spectrum {part[0]:.2f}, symmetry {part[1]:.3f}, transforms {part[2]:.2f}, mapping {part[3]:.2f} ms), "
        f"host-array call {float(np.mean(hms)):.1f} ms")
    if cpu:
        # the FP64 oracle on one core on a bounded sample (a 160^3 block of the same model parameters)
        cs = structured_cfg(n=(160, 160, 160), ds=c["ds"], acf=c["acf"], hurst=c["hurst"], cl=c["cl"],
                            sigma=c["sigma"], real=np.float32)
        t1 = time.perf_counter()
        r = fo.realization(dict(cs, method=0, pad=0, structured=True), c["seed"], np.float32)
        secs = time.perf_counter() - t1
        ni = int(np.prod(r["setup"]["npts"]))
        out["cpu_baseline"] = {"value": _sig(ni / secs / 1e6), "unit": "internal Mpt/s", "cores": 1, "kind": "port",
                               "sample": f"160^3 grid (internal {r['setup']['npts']}), FP64 numpy restatement "
                                         f"({secs:.1f} s)"}
    return out


def _host_threads():
    """Every core this process may run on (its affinity set)."""
    return len(os.sched_getaffinity(0))


def cpu_baseline(oracle, cfg, seed, flavour="f", threads=None, seconds_target=15.0):
    """The reference loop (harmonic outer, points inner, libm sin/cos at
    `real` precision) on the host cores, each thread owning a block of
    z-slabs (or of points) like an MPI rank, over a bounded subset of the
    same workload: calibrated on a short run, then sized to about
    seconds_target."""
    import ctypes as C

    from oracle_lib import _DP  # the oracle's binding, loaded only for this leg

    p = oracle.params(cfg)
    s = oracle.setup(p, flavour)
    harm, used, _ = oracle.draw(p, s, seed, flavour)
    threads = threads or _host_threads()
    nh = int(used.sum())
    structured = cfg.get("structured", True)
    if structured:
        nx, ny, nz = cfg["fe"][0], cfg["fe"][1], cfg["fe"][2]
        unit, total = nx * ny, nz  # points per slab, slabs
    else:
        unit, total = 1, p.npts
    real = np.float32 if flavour == "f" else np.float64

    def run(nunits, nharm_used):
        u = used.copy()
        idx = np.flatnonzero(u)
        u[idx[nharm_used:]] = 0
        out = np.zeros(unit * nunits, dtype=real)
        t0 = time.perf_counter()
        if structured:
            fn = getattr(oracle.L, f"orc_baseline_structured_{flavour}")
            fn(C.byref(p), C.byref(s), harm.ctypes.data_as(_DP), u.ctypes.data_as(C.POINTER(C.c_uint8)), 0, nunits,
               out.ctypes.data_as(C.c_void_p), threads)
        else:
            fn = getattr(oracle.L, f"orc_baseline_unstructured_{flavour}")
            fn(C.byref(p), C.byref(s), harm.ctypes.data_as(_DP), u.ctypes.data_as(C.POINTER(C.c_uint8)), C.c_long(0),
               C.c_long(nunits), out.ctypes.data_as(C.c_void_p), threads)
        return time.perf_counter() - t0

    probe_units = min(total, threads if structured else 200_000)
    probe_h = min(nh, 200)
    tp = run(probe_units, probe_h)
    rate = unit * probe_units * probe_h / tp
    n_units = int(seconds_target * rate / (unit * nh))
    step = threads if structured else 1
    n_units = min(total, max(step, n_units // step * step))
    hh = nh
    if unit * n_units * nh / rate > 4 * seconds_target:  # even the smallest subset is too long: cut harmonics
        hh = max(probe_h, int(seconds_target * rate / (unit * n_units)))
    t = run(n_units, hh)
    wps = unit * n_units * hh / t
    what = f"{n_units} z-slabs of {nx}x{ny}" if structured else f"{n_units} points"
    return dict(value=wps / 1e9, unit="Gpt·harm/s", cores=threads, kind="port",
                nproc=os.cpu_count(), affinity=len(os.sched_getaffinity(0)),
                sample=f"{what} x {hh} harmonics ({t:.1f} s), reference loop order, "
                       f"{'FP32' if flavour == 'f' else 'FP64'} libm sin/cos, {threads} OpenMP thread(s) each owning "
                       f"{'z-slabs' if structured else 'a point range'}")


def oracle_points(oracle, cfg, seed, flavour, nsamp=256):
    """FP64 CPU oracle at sampled points of the workload (same draw as the
    library): returns (flat indices, values)."""
    p = oracle.params(cfg)
    s = oracle.setup(p, flavour)
    harm, used, _ = oracle.draw(p, s, seed, flavour)
    rng = np.random.default_rng(5)
    if cfg.get("structured", True):
        n = [cfg["fe"][a] - cfg["fs"][a] + 1 for a in range(3)]
        ii, jj, kk = (rng.integers(0, n[a], nsamp) for a in range(3))
        ref = oracle.field_at(p, s, harm, used, ii, jj, kk)
        return ii + n[0] * (jj + n[1] * kk), ref
    flat = rng.integers(0, p.npts, nsamp)
    sub = dict(cfg, x=cfg["x"][flat], y=cfg["y"][flat], z=cfg["z"][flat])
    p2 = oracle.params(sub)  # same parameters, the sampled points only
    return flat, oracle.field_unstructured(p2, s, harm, used)


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="precision_512", choices=sorted(WORKLOADS) + ["ensemble_64", "copy_calib", "fim_500"])
    ap.add_argument("--kernel", default=None, choices=KERNELS, help="timed kernel (default: the workload's)")
    ap.add_argument("--no-compare", action="store_true", help="skip the comparison kernels and the FP64 reference")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-e2e", action="store_true", help="skip the end-to-end scarf_execute timings")
    ap.add_argument("--no-ensemble", action="store_true", help="skip the 64-member ensemble (default workload)")
    ap.add_argument("--no-fim", action="store_true", help="skip the FIM (method 0) timing (default workload)")
    args = ap.parse_args(argv)
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the SRM shards by z-slab ranges with no exchange inside the harmonic "
              "loop, and multi-GPU runs are not implemented; run with --gpus 1", file=sys.stderr)
        return 2

    if args.workload == "ensemble_64":
        args.kernel = args.kernel or "mfma_bf16x3"
        return bench_ensemble(args)
    if args.workload == "copy_calib":
        return bench_copy_calibration(args)
    if args.workload == "fim_500":
        f = measure_fim(args.steps, args.warmup, cpu=not args.no_cpu)
        out = {"metric": "FIM realizations: 500^3 grid (reference examples), external Mpt/s", "value": f["mpts_per_s"],
               "unit": "Mpt/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": f["ms"],
               "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp32",
               "data": "synthetic", "config": {k: v for k, v in f.items() if k not in ("hbm", "cpu_baseline")},
               "roofline": {"bound": "hbm", "achieved": f["hbm"]["achieved_gbs"], "peak": PEAK_HBM_GBS,
                            "unit": "GB/s", "frac": f["hbm"]["frac"], "traffic": None, "kernel": "whole FIM pass"},
               "cpu_baseline": f.get("cpu_baseline")}
        print(json.dumps(out), flush=True)
        return 0

    import scarf3d_amd
    from oracle_lib import Oracle, epilogue_at
    from scarf3d_amd.hip import Hip

    w = WORKLOADS[args.workload]
    kernel = args.kernel or w["kernel"]
    flavour = w["flavour"]
    real = np.float32 if flavour == "f" else np.float64
    lib = scarf3d_amd.load(flavour)
    cfg = init(lib, w)
    structured = cfg.get("structured", True)
    npts = int(np.prod(w["n"])) if structured else int(w["points"])
    work = float(npts) * w["nharm"]
    e2e = None
    if not args.no_e2e:
        e2e = measure_end_to_end(lib, w, kernel, max(3, min(args.steps, 10)), 2)
    hip = Hip()
    d_field = hip.empty(npts, real)
    n_used, host_s = lib.srm_draw(w["seed"])
    shape = w["n"] if structured else f"{npts} points"
    log(f"[bench] {args.workload}: {shape} x {w['nharm']} harmonics ({n_used} kept), host draw {host_s:.3f} s")

    res = {kernel: time_kernel(lib, hip, kernel, d_field, args.steps, args.warmup)}
    tile = lib.last_tile() if kernel.startswith("mfma") else None
    main_field = d_field.numpy()
    log(f"[bench] {kernel}: {res[kernel]['field_ms']:.3f} ms field kernel, {res[kernel]['ms_per_step']:.3f} ms/step")

    extra = {}
    if not args.no_compare:
        for k in w["compare"]:
            if k == kernel:
                continue
            slow = k in ("direct_f32", "direct_f64") and work > 1e12
            steps = max(1, min(3, args.steps)) if slow else args.steps
            res[k] = time_kernel(lib, hip, k, d_field, steps, 1)
            log(f"[bench] {k}: {res[k]['field_ms']:.3f} ms field kernel")
            res[k]["field"] = d_field.numpy()
        d_field.free()
        # FP64 reference over the whole field, on the same resident table
        t0 = time.perf_counter()
        d_ref = hip.empty(npts, np.float64)
        st64 = lib.srm_run_fp64(d_ref.ptr)  # {count, mean, variance, sqrt} of the field before the epilogue
        hip.synchronize()
        ref64 = d_ref.numpy()
        d_ref.free()
        log(f"[bench] FP64 reference field in {time.perf_counter() - t0:.1f} s")
        sigma = cfg["sigma"]
        res[kernel]["field"] = main_field
        errs = {}
        for k, r in res.items():
            dif = r["field"].astype(np.float64) - ref64
            st3 = float(r["stats"][2])
            mx, rms = float(np.abs(dif).max()), float(np.sqrt(np.mean(dif * dif)))
            errs[k] = dict(max_err_sigma=mx / sigma, rms_err_sigma=rms / sigma, max_err_stats3=mx / st3)
            del dif
            log(f"[bench] {k}: max|err| = {errs[k]['max_err_sigma']:.2e} sigma, rms {errs[k]['rms_err_sigma']:.2e}")
        # the FP64 kernel and the timed kernel against the CPU oracle at sampled points (same draw)
        flat, ref_pts = oracle_points(Oracle(), cfg, w["seed"], flavour)
        ref_pts = epilogue_at(ref_pts, flat, cfg, st64[1], st64[2])
        extra["oracle_points"] = dict(
            n=len(flat), note="FP64 CPU oracle vs the timed kernel's field at sampled points (same draw)",
            max_err_sigma=float(np.abs(main_field[flat].astype(np.float64) - ref_pts).max() / sigma))
        extra["fp64_kernel_vs_oracle_max_err_sigma"] = float(np.abs(ref64[flat] - ref_pts).max() / sigma)
        log(f"[bench] oracle points: {extra['oracle_points']['max_err_sigma']:.2e} sigma; FP64 kernel vs oracle "
            f"{extra['fp64_kernel_vs_oracle_max_err_sigma']:.2e} sigma")
        del ref64
        for k in res:
            res[k].pop("field", None)
            res[k].update(errs.get(k, {}))
    else:
        d_field.free()

    main_r = res[kernel]
    P = MFMA_PRODUCTS.get(kernel)
    if P:
        achieved = work * 4 * P / (main_r["field_ms"] * 1e-3) / 1e12
        roof = {"bound": "mfma", "achieved": _sig(achieved), "peak": PEAK_MFMA_TFLOPS, "unit": "TFLOP/s",
                "frac": _sig(achieved / PEAK_MFMA_TFLOPS), "traffic": None,
                "kernel": f"mfma_grid<{kernel}>", "flops_per_point_harmonic": 4 * P,
                "useful_frac": _sig(work * 4 / (main_r["field_ms"] * 1e-3) / 1e12 / PEAK_MFMA_TFLOPS)}
    elif kernel == "direct_f64":
        achieved = work * 10 / (main_r["field_ms"] * 1e-3) / 1e12
        roof = {"bound": "valu", "achieved": _sig(achieved), "peak": PEAK_VALU_F64_TFLOPS, "unit": "TFLOP/s",
                "frac": _sig(achieved / PEAK_VALU_F64_TFLOPS), "traffic": None,
                "kernel": "direct_grid_f64" if structured else "direct_points<f64>", "flops_per_point_harmonic": 10}
    else:
        achieved = work * 10 / (main_r["field_ms"] * 1e-3) / 1e12
        roof = {"bound": "valu", "achieved": _sig(achieved), "peak": PEAK_VALU_TFLOPS, "unit": "TFLOP/s",
                "frac": _sig(achieved / PEAK_VALU_TFLOPS), "traffic": None,
                "kernel": "direct_grid_f32" if structured else "direct_points<f32>", "flops_per_point_harmonic": 10}

    if (args.workload, kernel) in TRAFFIC and tile is not None and tile[0] == 128:
        roof["traffic"], roof["traffic_source"] = TRAFFIC[(args.workload, kernel)]
    cpu = None
    if not args.no_cpu:
        oracle = Oracle()
        cpu = cpu_baseline(oracle, cfg, w["seed"], flavour)
        log(f"[bench] CPU baseline {cpu['value']:.4f} Gpt.harm/s on {cpu['cores']} threads ({cpu['sample']})")
        one = cpu_baseline(oracle, cfg, w["seed"], flavour, threads=1,
                           seconds_target=15.0 if w.get("cpu_one_rank") else 8.0)
        extra["cpu_baseline_one_core"] = one
        log(f"[bench] CPU baseline, one core: {one['value']:.4f} Gpt.harm/s ({one['sample']})")

    value = work / (main_r["ms_per_step"] * 1e-3) / 1e9
    dtype = {"mfma_bf16x3": "bf16x3-split MFMA, fp32 accumulate", "mfma_f16x2": "fp16x2-split (scaled) MFMA, fp32 "
             "accumulate", "mfma_bf16x2": "bf16x2-split MFMA, fp32 accumulate", "direct_f32": "f32 (FP64 phase "
             "reduction)", "direct_f64": "f64"}[kernel]
    config = {"workload": args.workload, "harmonics": w["nharm"], "dh_m": w["ds"],
              "acf": "von Karman" if w["acf"] == 0 else "Gaussian", "cl_m": list(w["cl"]), "sigma": w["sigma"],
              "seed": w["seed"], "kernel": kernel, "library": "libscarf3df" if flavour == "f" else "libscarf3d",
              "host_draw_s": _sig(host_s)}
    if tile:
        config["block_tile"] = dict(zip(("x", "j", "k"), tile))
    if structured:
        config["grid"] = list(w["n"])
    else:
        config["points"] = npts
        config["box_m"] = list(w["box"])
    if w["acf"] == 0:
        config["hurst"] = w["hurst"]
    out = {
        "metric": METRIC, "value": round(value, 2), "unit": "Gpt·harm/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": _sig(main_r["ms_per_step"]), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": dtype,
        "data": "synthetic (harmonics drawn on the host from the configured spectrum)",
        "config": config,
        "roofline": roof,
        "cpu_baseline": cpu,
        "kernels": {k: {kk: (_sig(vv) if isinstance(vv, float) else vv) for kk, vv in r.items() if kk != "stats"}
                    for k, r in res.items()},
    }
    if args.workload != "precision_512":
        out["metric"] = f"SRM Gpt·harm/s, workload {args.workload}"
    if "direct_f32" in res and kernel != "direct_f32":
        out["speedup_vs_fp32_direct"] = _sig(res["direct_f32"]["field_ms"] / main_r["field_ms"])
    for k, r in out["kernels"].items():
        rate = work / (r["field_ms"] * 1e-3)  # point-harmonics per second
        r.setdefault("gpt_harm_per_s", _sig(rate / 1e9))
        if "direct_f32" in res and k != "direct_f32":
            r["speedup_vs_fp32_direct"] = _sig(res["direct_f32"]["field_ms"] / r["field_ms"])
        # two rooflines: the reference formulation's 10 FP32 flops per
        # point-harmonic against the FP32 vector peak, and the executed MFMA flops
        # (4 per product per point-harmonic) against dense bf16/fp16
        r["frac_fp32_valu"] = _sig(rate * 10 / (PEAK_VALU_TFLOPS * 1e12))
        if k in MFMA_PRODUCTS:
            r["frac_bf16_mfma"] = _sig(rate * 4 * MFMA_PRODUCTS[k] / (PEAK_MFMA_TFLOPS * 1e12))
    out.update(extra)
    if e2e:
        # the reference's call, scarf_execute, warm: draw + device + copy into the host array
        ex = e2e["execute_streamed"]
        out["end_to_end_ms"] = _sig(ex["ms"])
        out["e2e_gpt_harm_per_s"] = _sig(work / (ex["ms"] * 1e-3) / 1e9)
        whole_draw = e2e["execute_whole_table"]["draw_ms"]
        e2e["device_ms"] = main_r["device_ms"]  # the same realization with its table resident
        e2e["max_draw_device_ms"] = max(whole_draw, main_r["device_ms"])
        e2e["note"] = ("ms per call, wall clock; draw_ms = the host draw inside the call; the streamed call "
                       "queues each chunk's device work while the next chunk is drawn")
        out["end_to_end"] = {k: ({kk: _sig(vv) for kk, vv in v.items()} if isinstance(v, dict) else
                                 (_sig(v) if isinstance(v, float) else v)) for k, v in e2e.items()}
    lib.finalize()
    if args.workload == "precision_512" and not args.no_ensemble:
        e = measure_ensemble("mfma_bf16x3", max(3, min(args.steps, 10)), 2)
        single = out["kernels"].get("mfma_bf16x3", {}).get("frac_bf16_mfma")
        out["ensemble_64"] = {
            "kernel": "mfma_bf16x3", "members": e["members"], "point_harmonics": e["work"], "ms": _sig(e["ms"]),
            "gpt_harm_per_s": _sig(e["work"] / (e["ms"] * 1e-3) / 1e9), "achieved_tflops": _sig(e["achieved"]),
            "frac": _sig(e["frac"]), "single_field_frac": single,
            "gap_to_single_field": _sig(1.0 - e["frac"] / single) if single else None,
            "first_run_s": _sig(e["first_s"]), "ms_per_call_wall": _sig(e["wall_ms"]),
            "note": "one persistent grouped-GEMM launch per realization set, replayed from a hipGraph; ms = device "
                    "time of the replay (HIP events), frac against 2.5 PFLOP/s dense bf16 at 24 flop per "
                    "point-harmonic"}
    if args.workload == "precision_512" and not args.no_fim:
        out["fim_500"] = measure_fim(max(3, min(args.steps, 10)), 1, cpu=not args.no_cpu)
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
