"""Benchmark: (k, omega) surface Green's function solves per second at Ndim = 72.

Workload (one step = one pass of the hot path over the whole grid): the
36-orbital synthetic model (R in [-3,3]^3, 343 R vectors, seed 2), Np = 2
principal layers (Ndim = 72), 512 k points on the (-0.5,0)->(0.5,0) path x 512
energies on [-1, 1) eV = 262,144 instances, eta = 1e-3 eV, the reference
decimation stop rule (sum |alpha| <= 1e-16 Ha, itermax 100).  Inputs (model,
k points, energies) are resident on the device before timing starts; a step
is the Fourier sum plus the batched decimation and traces.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--precision fp64|fp32|auto]
    python bench.py --workload plane288|mixed|c1 [--steps K] [--warmup W]
    python bench.py --summarize-rocprof [plane288|plane384] TRACE_DIR FETCH_DIR WRITE_DIR COPY_FETCH_DIR COPY_WRITE_DIR
    python bench.py --summarize-trace TRACE_DIR KERNEL [KERNEL ...]
    python bench.py --summarize-counters PMC_DIR KERNEL [KERNEL ...]

Prints one JSON line.  The decimation runs as rounds of two kernels on two
streams (mid_inverse_kernel and mid_gemm_kernel); the roofline figures refer to
that whole decimation stage, timed with HIP events on the first stream, which
waits for the second at the end of the stage.  --summarize-rocprof turns the
rocprofv3 runs of the same command (kernel trace; FETCH_SIZE and WRITE_SIZE
counters; the same counters on a plain 1 GiB copy for calibration) into the
summary kept under profiles/.  The FP64 path always runs (it defines the per-instance
reference iteration count I_ref used for the algorithmic flop count
F = (56 I_ref + 24) N^3 per solve).  The reported `value` is the solves/s of
the fastest path whose A(k, omega) error against FP64 is <= 1e-6.

Three more workloads, FP64 only, print a line of the same form:
  c1        the 8-orbital model (Ndim = 16, R in {-1,0,1}^3), 201 k x 401
            energies on the same path and window, eta = 1e-3 eV;
  plane288  the 144-orbital spinful model (Ndim = 288, R in [-3,3]^3) on an
            nk x nk sampling (default 257 x 257, the reference's rounding of
            256 x 256) of the k-plane [-0.5, 0.5]^2 at
            omega = 0, eta = 5e-4 eV, traces divided by pi (SurfaceDOSkk);
  mixed     four models (Num_wann, Np) = (8, 1), (16, 2), (36, 3), (72, 3)
            (Ndim 8, 32, 108, 216; R in [-2,2]^3), 25,000 instances each with
            k from 500 random points, omega uniform on [-1, 1] eV and eta
            log-uniform on [1e-4, 1e-2] eV, through the per-instance batch
            entry point (its small per-instance arrays are uploaded and the
            traces downloaded inside each step).
--summarize-trace prints the kernel table and stage span of a rocprofv3
kernel trace of either; --summarize-counters the per-kernel sums of a
rocprofv3 --pmc run.
"""
from __future__ import annotations

import argparse
import json
import multiprocessing as mp
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

from wannier_tools_amd import model as M  # noqa: E402

TRAFFIC_JSON = "decimation_fp64_ndim72_512x512.traffic.json"
DECIMATION_KERNELS = ("mid_inverse_kernel", "mid_gemm_kernel")
LARGE_KERNELS = ("gj_large_round_kernel", "gemm_large_round_kernel")
# per workload: traffic file under profiles/, the stage's kernels, what was run
TRAFFIC = {
    "grid72": (TRAFFIC_JSON, DECIMATION_KERNELS, "decimation rounds (mid_inverse_kernel + "
               "mid_gemm_kernel)", "ndim72 512x512 eta=1e-3 eV"),
    "plane288": ("decimation_fp64_ndim288_kplane65.traffic.json", LARGE_KERNELS,
                 "decimation rounds (gj_large_round_kernel + gemm_large_round_kernel)",
                 "ndim288 65x65 k-plane omega=0 eta=5e-4 eV"),
    "plane288_257": ("decimation_fp64_ndim288_kplane257.traffic.json", LARGE_KERNELS,
                     "decimation rounds (gj_large_round_kernel + gemm_large_round_kernel)",
                     "ndim288 257x257 k-plane omega=0 eta=5e-4 eV"),
    "plane384": ("decimation_fp64_ndim384_kplane45.traffic.json", LARGE_KERNELS,
                 "decimation rounds (gj_large_round_kernel + gemm_large_round_kernel)",
                 "ndim384 45x45 k-plane omega=0 eta=5e-4 eV (--plane-nw 192 --nk 45)"),
}
FP64_MFMA_PEAK_TFLOPS = 78.6
FP32_MFMA_PEAK_TFLOPS = 157.3
HBM_PEAK_GBS = 8000.0
NW, NP_ = 36, 2
NDIM = NW * NP_


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def workload(nk: int, nomega: int):
    mdl = M.model_ndim72()
    irvec, hr = mdl.surface_cell()
    kpts = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], nk)
    omegas = M.omega_grid(-1.0, 1.0, nomega) * M.EV2HARTREE
    eta = 1e-3 * M.EV2HARTREE
    return irvec, hr, kpts, omegas, eta


PLANE_NW, PLANE_NP = 144, 2
PLANE_ETA_EV = 5e-4
MIXED_MODELS = ((8, 1, 40), (16, 2, 41), (36, 3, 42), (72, 3, 43))  # (Num_wann, Np, seed)
MIXED_PER_MODEL = 25000


def workload_plane288(nk: int, nw: int = 144):
    # nw = 144 is the named model; other sizes use the same recipe (R in
    # [-3, 3]^3, spinful, seed 5) to time the kernels at other orders
    mdl = M.model_ndim288() if nw == 144 else M.synthetic_model(
        nw, 3, 0.5, M.decay_l2(1.5), seed=5, soc_sigma=0.05, name=f"nw{nw}_soc_r3")
    irvec, hr = mdl.surface_cell()
    kpts, _, _ = M.kplane_slab((-0.5, -0.5), (1.0, 0.0), (0.0, 1.0), nk, nk)
    return irvec, hr, kpts, np.array([0.0]), PLANE_ETA_EV * M.EV2HARTREE


def workload_mixed(per_model: int):
    rng = np.random.default_rng(4)
    sets = []
    for nw, np_, seed in MIXED_MODELS:
        irvec, hr = M.synthetic_model(nw, 2, 0.5, M.decay_l2(1.5), seed=seed).surface_cell()
        sets.append(dict(nw=nw, np=np_, irvec=irvec, hr=hr,
                         kpts=rng.uniform(-0.5, 0.5, (500, 2)),
                         k_index=rng.integers(0, 500, per_model).astype(np.int32),
                         omega=rng.uniform(-1.0, 1.0, per_model) * M.EV2HARTREE,
                         eta=10.0 ** rng.uniform(-4.0, -2.0, per_model) * M.EV2HARTREE))
    return sets


def time_path(gf, precision: str, steps: int, warmup: int, divisor: float = 1.0):
    for i in range(warmup):
        gf.run_async(gf.eta, divisor, precision)
        gf.sync()
        log(f"[bench] {precision} warmup {i + 1}/{warmup}: decimation {gf.timing()[1]:.1f} ms")
    dec_ms = []
    t0 = time.perf_counter()
    for i in range(steps):
        gf.run_async(gf.eta, divisor, precision)
        gf.sync()
        dec_ms.append(gf.timing()[1])
        log(f"[bench] {precision} step {i + 1}/{steps}: decimation {dec_ms[-1]:.1f} ms")
    t1 = time.perf_counter()
    out = gf.download()
    return (t1 - t0) / steps, float(np.mean(dec_ms)), out


def alg_flops(ndim: int, iters) -> float:
    """F = (56 I_ref + 24) N^3 summed over the instances."""
    return float(np.sum(56.0 * np.asarray(iters, dtype=np.float64) + 24.0)) * float(ndim) ** 3


# ---- CPU baseline: the reference's own Fortran (oracle/_ref) or the C port --
def _cpu_worker(args):
    """Solve the jobs (model, k1, k2, omega, eta) in order, one H00/H01 per
    run of equal (model, k), as the reference's k-outer loops do."""
    kind, models, jobs = args
    os.environ["OPENBLAS_NUM_THREADS"] = "1"
    import oracle
    eng = oracle.RefHarness() if kind == "reference" else oracle.Oracle()
    cur_m, key, h = None, None, None
    for m, k1, k2, w, e in jobs:
        nw, np_, irvec, hr = models[m]
        if kind == "reference" and m != cur_m:
            eng.set_model(nw, np_, irvec, hr)
            cur_m = m
        if (m, k1, k2) != key:
            k = np.array([k1, k2])
            h = eng.ham_qlayer2qlayer(k) if kind == "reference" else \
                eng.ham_qlayer2qlayer(nw, np_, irvec, hr, k)
            key = (m, k1, k2)
        eng.surfgreen_1985(w, e, h[0], h[1])
    return len(jobs)


def _usable_cores() -> int:
    """Cores this process may run on (its affinity mask)."""
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:
        return os.cpu_count() or 1


def default_cpu_workers() -> int:
    """One CPU-baseline worker per usable core, capped by OMP_NUM_THREADS when
    the environment sets it (a shared host's CPU share for this job)."""
    n = _usable_cores()
    try:
        cap = int(os.environ.get("OMP_NUM_THREADS", "0"))
    except ValueError:
        cap = 0
    return max(1, min(n, cap) if cap > 0 else n)


def cpu_baseline(models, jobs, workers: int, what: str):
    """Time the reference CPU path on a bounded sample: `jobs` dealt
    round-robin over `workers` processes (the reference's MPI k round-robin),
    one OpenBLAS thread each."""
    import oracle
    kind = "reference" if oracle.ref_available() else "port"
    chunks = [sorted(jobs[w::workers], key=lambda j: (j[0], j[1], j[2])) for w in range(workers)]
    ctx = mp.get_context("spawn")
    os.environ["OPENBLAS_NUM_THREADS"] = "1"
    with ctx.Pool(workers) as pool:
        t0 = time.perf_counter()
        done = sum(pool.map(_cpu_worker, [(kind, models, c) for c in chunks]))
        dt = time.perf_counter() - t0
    return {
        "value": done / dt,
        "unit": "solves/s",
        "cores": workers,
        "host_cores": os.cpu_count(),
        "usable_cores": _usable_cores(),
        "kind": kind,
        "sample": (f"{done} {what}, "
                   f"{'reference ham_qlayer2qlayer + surfgreen_1985 (Fortran, OpenBLAS)' if kind == 'reference' else 'C FP64 restatement'}"
                   f", {workers} processes x 1 thread, {dt:.1f} s"),
    }


def grid_jobs(kpts, omegas, eta, total: int):
    """`total` (k, omega) instances evenly strided over the grid."""
    nk, nom = kpts.shape[0], omegas.size
    flat = np.linspace(0, nk * nom - 1, total).astype(np.int64)
    return [(0, float(kpts[t // nom, 0]), float(kpts[t // nom, 1]), float(omegas[t % nom]), eta)
            for t in flat]


def _csv_rows(d: str, suffix: str):
    import csv
    import glob
    paths = glob.glob(os.path.join(d, "**", "*" + suffix), recursive=True)
    if not paths:
        raise SystemExit(f"no *{suffix} under {d}")
    with open(paths[0]) as f:
        return list(csv.DictReader(f))


def _counter_kib(d: str, counter: str, kernels) -> float:
    """Sum of a rocprofv3 counter over the dispatches of the named kernels (KiB)."""
    return sum(float(r["Counter_Value"]) for r in _csv_rows(d, "counter_collection.csv")
               if r["Counter_Name"] == counter and any(k in r["Kernel_Name"] for k in kernels))


def _db_trace(d: str):
    """(stats, rows) of a rocprofv3 kernel trace written in its default SQLite
    (rocpd) form, shaped like the kernel_stats.csv / kernel_trace.csv rows."""
    import glob
    import sqlite3
    paths = glob.glob(os.path.join(d, "**", "*_results.db"), recursive=True)
    if not paths:
        return None
    con = sqlite3.connect(paths[0])
    rows = [{"Kernel_Name": n, "Start_Timestamp": s, "End_Timestamp": e}
            for n, s, e in con.execute("select name, start, end from kernels")]
    agg: dict = {}
    for r in rows:
        c, t = agg.get(r["Kernel_Name"], (0, 0))
        agg[r["Kernel_Name"]] = (c + 1, t + r["End_Timestamp"] - r["Start_Timestamp"])
    stats = [{"Name": n, "Calls": c, "TotalDurationNs": t, "AverageNs": t / c}
             for n, (c, t) in sorted(agg.items(), key=lambda kv: -kv[1][1])]
    con.close()
    return stats, rows


def _trace_table(trace, kernels, rows_shown: int = 8):
    """Kernel table of a rocprofv3 kernel trace (CSV or SQLite output), and the
    span (first start to last end) and busy time of the dispatches whose names
    contain `kernels`."""
    db = _db_trace(trace)
    if db is not None:
        stats, rows = db
    else:
        stats = _csv_rows(trace, "kernel_stats.csv")
        rows = _csv_rows(trace, "kernel_trace.csv")
    sel = [r for r in rows if any(k in r["Kernel_Name"] for k in kernels)]
    if not sel:
        raise SystemExit(f"no dispatch of {kernels} in {trace}")
    span_ns = max(int(r["End_Timestamp"]) for r in sel) - min(int(r["Start_Timestamp"]) for r in sel)
    busy = {k: sum(int(r["End_Timestamp"]) - int(r["Start_Timestamp"]) for r in sel
                   if k in r["Kernel_Name"]) for k in kernels}
    print("| Kernel | Calls | Total ms | Average us |\n|---|---|---|---|")
    for r in stats[:rows_shown]:
        print(f"| `{r['Name'][:90]}` | {r['Calls']} | {float(r['TotalDurationNs']) / 1e6:.1f} | "
              f"{float(r['AverageNs']) / 1e3:.1f} |")
    print(f"\nSpan of the {', '.join(kernels)} dispatches (first start to last end): "
          f"{span_ns / 1e6:.1f} ms; " + "; ".join(f"{k} busy {v / 1e6:.1f} ms" for k, v in busy.items()))
    return span_ns


def summarize_counters(d, *kernels) -> int:
    """Per kernel (dispatches whose names contain each of `kernels`) of a
    rocprofv3 --pmc run (CSV): dispatch count, summed and mean dispatch time
    (the counter run serialises dispatches, so these are times alone), and
    every counter summed over the dispatches."""
    rows = _csv_rows(d, "counter_collection.csv")
    print("| Kernel | Dispatches | Total ms | Mean us | Counter | Sum |\n|---|---|---|---|---|---|")
    for k in kernels:
        sel = [r for r in rows if k in r["Kernel_Name"]]
        if not sel:
            raise SystemExit(f"no dispatch of {k} in {d}")
        dur = {r["Dispatch_Id"]: int(r["End_Timestamp"]) - int(r["Start_Timestamp"]) for r in sel}
        sums: dict = {}
        for r in sel:
            sums[r["Counter_Name"]] = sums.get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
        tot = sum(dur.values())
        for i, (c, v) in enumerate(sorted(sums.items())):
            head = (f"| `{k}` | {len(dur)} | {tot / 1e6:.2f} | {tot / len(dur) / 1e3:.1f} "
                    if i == 0 else "| | | | ")
            print(f"{head}| {c} | {v:.4e} |")
    return 0


def summarize_trace(trace, *kernels) -> int:
    """Kernel table and span of a rocprofv3 kernel trace (any workload)."""
    _trace_table(trace, kernels, rows_shown=12)
    return 0


def summarize_rocprof(*argv) -> int:
    """profiles/ summary of the decimation stage from rocprofv3 runs of
    `bench.py --steps 1 --warmup 0 --no-cpu-baseline --precision fp64` (or of
    `--workload plane288` when the first argument names it): arguments
    [WORKLOAD] TRACE FETCH WRITE COPY_FETCH COPY_WRITE."""
    workload = argv[0] if len(argv) == 6 else "grid72"
    trace, fetch, write, cfetch, cwrite = argv[-5:]
    fname, kernels, stage, what = TRAFFIC[workload]
    span_ns = _trace_table(trace, kernels)
    # counter scale: KiB reported for a copy of known size
    copy_bytes = 1 << 30
    f_scale = copy_bytes / (_counter_kib(cfetch, "FETCH_SIZE", ("copyBuffer",)) * 1024)
    w_scale = copy_bytes / (_counter_kib(cwrite, "WRITE_SIZE", ("copyBuffer",)) * 1024)
    fetch_b = _counter_kib(fetch, "FETCH_SIZE", kernels) * 1024 * f_scale
    write_b = _counter_kib(write, "WRITE_SIZE", kernels) * 1024 * w_scale
    json.dump({"stage": stage, "workload": what, "fetch_bytes": fetch_b,
               "write_bytes": write_b, "fetch_scale": f_scale, "write_scale": w_scale,
               "span_ns": span_ns}, open(os.path.join(ROOT, "profiles", fname), "w"),
              indent=1)
    print(f"\nHBM traffic of the stage: fetch {fetch_b:.4e} B (scale {f_scale:.3f}), "
          f"write {write_b:.4e} B (scale {w_scale:.3f}), {(fetch_b + write_b) / span_ns:.1f} GB/s "
          f"over the span")
    return 0


def run_grid72(args, SurfaceGF) -> dict:
    """The Ndim = 72 k-path x energy grid (the headline line)."""
    irvec, hr, kpts, omegas, eta = workload(args.nk or 512, args.nomega or 512)
    ninst = kpts.shape[0] * omegas.size
    gf = SurfaceGF(0)
    gf.set_model_arrays(NW, NP_, irvec, hr)
    gf.upload_grid(kpts, omegas)
    gf.eta = eta
    # auxiliary paths (other schedules and precisions) are timed over at most
    # three steps after one warmup step: their step times vary by well under 1%
    aux_steps, aux_warmup = min(args.steps, 3), min(args.warmup, 1)
    scheds = ["persistent", "rounds"] if args.schedule == "both" else [args.schedule]
    sched_res = {}
    for sch in scheds[:-1]:  # the last one is timed below in full and kept
        gf.set_schedule(sch)
        log(f"[bench] FP64 path, {sch} schedule: {ninst} instances, Ndim={NDIM}")
        s_, d_, o_ = time_path(gf, "fp64", aux_steps, aux_warmup)
        sched_res[sch] = {"s_per_step": s_, "solves_per_s": ninst / s_, "decimate_ms": d_,
                          "steps": aux_steps}
    gf.set_schedule(scheds[-1])
    gf.upload_grid(kpts, omegas)

    log(f"[bench] FP64 path, {scheds[-1]} schedule: {ninst} instances, Ndim={NDIM}")
    s64, dec64, out64 = time_path(gf, "fp64", args.steps, args.warmup)
    sched_res[scheds[-1]] = {"s_per_step": s64, "solves_per_s": ninst / s64, "decimate_ms": dec64}
    dl64, dr64, db64, it64, st64 = out64
    flops = alg_flops(NDIM, it64)
    res = {
        "fp64": {"s_per_step": s64, "solves_per_s": ninst / s64, "decimate_ms": dec64,
                 "mean_iters": float(it64.mean()), "max_iters": int(it64.max()),
                 "not_converged": int(np.count_nonzero(st64 & 2)),
                 "singular": int(np.count_nonzero(st64 & 1)),
                 "mfma_tflops_algorithmic": flops / (dec64 * 1e-3) / 1e12,
                 "schedule": scheds[-1], "schedules": sched_res},
    }
    log(f"[bench] fp64: {ninst / s64:.1f} solves/s, {s64:.3f} s/step, decimation {dec64:.1f} ms")

    best = ("fp64", s64, dec64, FP64_MFMA_PEAK_TFLOPS)

    def error_report(d):
        rel = np.concatenate([np.abs(x - y).ravel() / np.abs(y).ravel() for x, y in
                              ((d[0], dl64), (d[1], dr64), (d[2], db64))])
        per_file = {}
        for name_, x, y in (("dos.dat_l", d[0], dl64), ("dos.dat_r", d[1], dr64),
                            ("dos.dat_bulk", d[2], db64)):
            r_ = (np.abs(x - y) / np.abs(y)).ravel()
            per_file[name_] = {"max_rel_err_A": float(r_.max()),
                               "median_rel_err_A": float(np.median(r_))}
        return {"max_rel_err_A": float(rel.max()), "median_rel_err_A": float(np.median(rel)),
                "frac_within_1e-6": float(np.mean(rel <= 1e-6)), "per_file": per_file}

    # FP32 working precision (measurement mode): speed and error on A against
    # the FP64 path (the mixed precision runs as FP64 and is not timed again)
    for prec, peak_ in (("fp32", FP32_MFMA_PEAK_TFLOPS),):
        if args.precision not in ("auto", prec):
            continue
        try:
            s_p, dec_p, out_p = time_path(gf, prec, aux_steps, aux_warmup)
        except Exception as e:  # path not available in this build
            log(f"[bench] {prec} unavailable: {e}")
            continue
        rep = error_report(out_p[:3])
        res[prec] = {"s_per_step": s_p, "solves_per_s": ninst / s_p, "decimate_ms": dec_p,
                     "steps": aux_steps, **rep, "speedup_vs_fp64": s64 / s_p,
                     "iterations_differing_from_fp64": int(np.count_nonzero(out_p[3] != it64))}
        log(f"[bench] {prec}: {ninst / s_p:.1f} solves/s, max rel err {rep['max_rel_err_A']:.2e}")
        if rep["max_rel_err_A"] <= 1e-6 and s_p < best[1]:
            best = (prec, s_p, dec_p, peak_)

    name, s_step, dec_ms, peak = best
    achieved = flops / (dec_ms * 1e-3) / 1e12
    # HBM bytes per launch of this kernel on this workload, from the committed
    # rocprofv3 FETCH_SIZE / WRITE_SIZE runs (scaled by a 1 GiB copy calibration)
    traffic = None
    tpath = os.path.join(ROOT, "profiles", TRAFFIC_JSON)
    if name == "fp64" and (kpts.shape[0], omegas.size) == (512, 512) and os.path.exists(tpath):
        t = json.load(open(tpath))
        traffic = t["fetch_bytes"] + t["write_bytes"]
    out = {
        "metric": "G(k,w) solves/s @Ndim=72: FP32+refine vs FP64 GPU, err<=1e-6; %MFMA peak",
        "value": ninst / s_step,
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": s_step * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp64": "c128", "fp32": "c64+c128"}[name],
        "data": "synthetic",
        "config": {"workload": "surface GF k-path x energy grid, 36-orbital synthetic model, Np=2",
                   "ndim": NDIM, "num_wann": NW, "np": NP_, "nr": int(irvec.shape[0]),
                   "nk": int(kpts.shape[0]), "nomega": int(omegas.size), "instances": ninst,
                   "eta_ev": 1e-3, "stop_rule": "sum|alpha|<=1e-16 Ha, itermax 100",
                   "path": name},
        "roofline": {"bound": "mfma", "achieved": achieved, "peak": peak, "unit": "TFLOP/s",
                     "frac": achieved / peak, "traffic": traffic,
                     "kernel": {"fp64": "decimation stage: mid_inverse_kernel<9> + "
                                         "mid_gemm_kernel<9> rounds on two streams",
                                "fp32": "decimation stage: gj_round_kernel<5, float> + "
                                        "gemm_round_kernel<5, float, true> rounds on two streams"}[name],
                     "flops_per_launch": flops},
        "paths": res,
    }
    gf.close()
    if not args.no_cpu_baseline:
        log("[bench] CPU baseline ...")
        total = (args.cpu_per_worker or 1200) * args.cpu_workers
        out["cpu_baseline"] = cpu_baseline([(NW, NP_, irvec, hr)],
                                           grid_jobs(kpts, omegas, eta, total), args.cpu_workers,
                                           f"(k, omega) instances strided over the "
                                           f"{kpts.shape[0]}x{omegas.size} grid")
    return out


def run_plane288(args, SurfaceGF) -> dict:
    """The Ndim = 288 model on a k-plane at omega = 0 (FP64)."""
    nk = args.nk or 257
    nw = args.plane_nw
    irvec, hr, kpts, omegas, eta = workload_plane288(nk, nw)
    ninst = kpts.shape[0]
    n = nw * PLANE_NP
    q = (n + 15) // 16
    gf = SurfaceGF(0)
    gf.set_model_arrays(nw, PLANE_NP, irvec, hr)
    gf.upload_grid(kpts, omegas)
    gf.eta = eta
    log(f"[bench] plane288: {ninst} instances, Ndim={n}")
    s, dec, res = time_path(gf, "fp64", args.steps, args.warmup, M.REF_PI)
    its, st = res[3], res[4]
    flops = alg_flops(n, its)
    gf.close()
    log(f"[bench] plane288: {ninst / s:.1f} solves/s, decimation {dec:.1f} ms")
    achieved = flops / (dec * 1e-3) / 1e12
    # HBM bytes of the stage on this workload, from the committed rocprofv3
    # FETCH_SIZE / WRITE_SIZE runs (scaled by a 1 GiB copy calibration)
    traffic = None
    key = {(65, PLANE_NW): "plane288", (45, 192): "plane384", (257, PLANE_NW): "plane288_257"}.get((nk, nw))
    tpath = os.path.join(ROOT, "profiles", TRAFFIC[key][0]) if key else ""
    if key and os.path.exists(tpath):
        t = json.load(open(tpath))
        traffic = t["fetch_bytes"] + t["write_bytes"]
    out = {
        "metric": f"G(k,w) solves/s @Ndim={n}, k-plane at omega=0 (FP64)",
        "value": ninst / s, "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": s * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "c128", "data": "synthetic",
        "config": {"workload": f"surface GF k-plane {nk}x{nk} over [-0.5,0.5]^2 at omega=0, "
                               f"{nw}-orbital spinful synthetic model, Np=2",
                   "ndim": n, "num_wann": nw, "np": PLANE_NP, "nr": int(irvec.shape[0]),
                   "nk": ninst, "instances": ninst, "eta_ev": PLANE_ETA_EV, "divisor": "pi",
                   "stop_rule": "sum|alpha|<=1e-16 Ha, itermax 100", "path": "fp64",
                   "mean_iters": float(its.mean()), "not_converged": int(np.count_nonzero(st & 2))},
        "roofline": {"bound": "mfma", "achieved": achieved, "peak": FP64_MFMA_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": achieved / FP64_MFMA_PEAK_TFLOPS, "traffic": traffic,
                     "kernel": f"decimation stage: gj_large_round_kernel<{q}, double> + "
                               f"gemm_large_round_kernel<{q}, double> rounds on two streams",
                     "flops_per_launch": flops},
    }
    if not args.no_cpu_baseline:
        log("[bench] CPU baseline ...")
        total = (args.cpu_per_worker or 18) * args.cpu_workers
        out["cpu_baseline"] = cpu_baseline([(nw, PLANE_NP, irvec, hr)],
                                           grid_jobs(kpts, omegas, eta, total), args.cpu_workers,
                                           f"k points strided over the {nk}x{nk} plane")
    return out


def run_c1(args, SurfaceGF) -> dict:
    """The Ndim = 16 k-path x energy grid: the 8-orbital synthetic model (R in
    {-1,0,1}^3, seed 1), Np = 2, 201 k on the (-0.5,0)->(0.5,0) path x 401
    energies on [-1, 1) eV, eta = 1e-3 eV (FP64, the small-order kernel)."""
    nk, nom = args.nk or 201, args.nomega or 401
    irvec, hr = M.model_ndim16().surface_cell()
    kpts = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], nk)
    omegas = M.omega_grid(-1.0, 1.0, nom) * M.EV2HARTREE
    eta = 1e-3 * M.EV2HARTREE
    ninst = nk * nom
    gf = SurfaceGF(0)
    gf.set_model_arrays(8, 2, irvec, hr)
    gf.upload_grid(kpts, omegas)
    gf.eta = eta
    log(f"[bench] c1: {ninst} instances, Ndim=16")
    s, dec, res = time_path(gf, "fp64", args.steps, args.warmup)
    its, st = res[3], res[4]
    flops = alg_flops(16, its)
    gf.close()
    log(f"[bench] c1: {ninst / s:.1f} solves/s, decimation {dec:.2f} ms")
    achieved = flops / (dec * 1e-3) / 1e12
    out = {
        "metric": "G(k,w) solves/s @Ndim=16, k-path x energy grid (FP64)",
        "value": ninst / s, "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": s * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "c128", "data": "synthetic",
        "config": {"workload": f"surface GF k-path x energy grid {nk}x{nom}, 8-orbital synthetic "
                               "model, Np=2", "ndim": 16, "num_wann": 8, "np": 2,
                   "nr": int(irvec.shape[0]), "nk": nk, "nomega": nom, "instances": ninst,
                   "eta_ev": 1e-3, "stop_rule": "sum|alpha|<=1e-16 Ha, itermax 100", "path": "fp64",
                   "mean_iters": float(its.mean()), "not_converged": int(np.count_nonzero(st & 2))},
        # the kernel runs on the vector ALUs, whose FP64 peak on MI355X equals
        # the FP64 matrix peak
        "roofline": {"bound": "mfma", "achieved": achieved, "peak": FP64_MFMA_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": achieved / FP64_MFMA_PEAK_TFLOPS, "traffic": None,
                     "kernel": "decimation stage: tiny16_kernel<4> (one wave per instance, "
                               "matrix cores and vector ALUs, FP64 peak 78.6 TFLOP/s each)",
                     "flops_per_launch": flops},
    }
    if not args.no_cpu_baseline:
        log("[bench] CPU baseline ...")
        total = (args.cpu_per_worker or 80000) * args.cpu_workers
        out["cpu_baseline"] = cpu_baseline([(8, 2, irvec, hr)], grid_jobs(kpts, omegas, eta, total),
                                           args.cpu_workers,
                                           f"(k, omega) instances strided over the {nk}x{nom} grid")
    return out


def run_mixed(args, SurfaceGF) -> dict:
    """Four models, per-instance (k, omega, eta), through the batch entry point (FP64)."""
    sets = workload_mixed(MIXED_PER_MODEL)
    ctxs = []
    for w in sets:
        gf = SurfaceGF(0)
        gf.set_model_arrays(w["nw"], w["np"], w["irvec"], w["hr"])
        ctxs.append(gf)

    def step():
        dec, outs = [], []
        for gf, w in zip(ctxs, sets):
            outs.append(gf.spectral_batch(w["kpts"], w["k_index"], w["omega"], w["eta"]))
            dec.append(gf.timing()[1])
        return dec, outs

    for i in range(args.warmup):
        step()
        log(f"[bench] mixed warmup {i + 1}/{args.warmup}")
    decs = []
    t0 = time.perf_counter()
    for i in range(args.steps):
        dec, outs = step()
        decs.append(dec)
        log(f"[bench] mixed step {i + 1}/{args.steps}: decimation "
            + ", ".join(f"{d:.1f}" for d in dec) + " ms")
    s = (time.perf_counter() - t0) / args.steps
    for gf in ctxs:
        gf.close()
    ninst = MIXED_PER_MODEL * len(sets)
    dec_ms = np.mean(np.array(decs), axis=0)
    flops_m = [alg_flops(w["nw"] * w["np"], o[3]) for w, o in zip(sets, outs)]
    flops = float(sum(flops_m))
    achieved = flops / (float(dec_ms.sum()) * 1e-3) / 1e12
    members = {f"ndim{w['nw'] * w['np']}": {
        "solves_per_s_device": MIXED_PER_MODEL / (d * 1e-3), "decimate_ms": float(d),
        "tflops_algorithmic": f / (d * 1e-3) / 1e12, "mean_iters": float(o[3].mean()),
        "not_converged": int(np.count_nonzero(o[4] & 2))}
        for w, d, f, o in zip(sets, dec_ms, flops_m, outs)}
    log(f"[bench] mixed: {ninst / s:.1f} solves/s")
    out = {
        "metric": "G(k,w) solves/s, mixed models Ndim 8-216, per-instance eta (FP64)",
        "value": ninst / s, "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": s * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "c128", "data": "synthetic",
        "config": {"workload": "surface GF per-instance batch: 4 synthetic models "
                               "(Num_wann, Np) = (8,1), (16,2), (36,3), (72,3), R in [-2,2]^3, "
                               f"{MIXED_PER_MODEL} instances each, eta log-uniform [1e-4, 1e-2] eV",
                   "instances": ninst, "stop_rule": "sum|alpha|<=1e-16 Ha, itermax 100",
                   "path": "fp64", "members": members},
        "roofline": {"bound": "mfma", "achieved": achieved, "peak": FP64_MFMA_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": achieved / FP64_MFMA_PEAK_TFLOPS, "traffic": None,
                     "kernel": "decimation stages of the four models: tiny4_kernel<2> (Ndim 8), "
                               "small_kernel (32; vector ALUs), mid_inverse_kernel<14> + mid_gemm_kernel<14> "
                               "(108 padded to 112), gj_large_round_kernel<14, double> + "
                               "gemm_large_round_kernel<14, double> (216 padded to 224)",
                     "flops_per_launch": flops},
    }
    if not args.no_cpu_baseline:
        log("[bench] CPU baseline ...")
        per = args.cpu_per_worker or 60
        models, jobs = [], []
        for m, w in enumerate(sets):
            models.append((w["nw"], w["np"], w["irvec"], w["hr"]))
            pick = np.linspace(0, MIXED_PER_MODEL - 1, per * args.cpu_workers).astype(np.int64)
            jobs += [(m, float(w["kpts"][w["k_index"][i], 0]), float(w["kpts"][w["k_index"][i], 1]),
                      float(w["omega"][i]), float(w["eta"][i])) for i in pick]
        out["cpu_baseline"] = cpu_baseline(models, jobs, args.cpu_workers,
                                           "instances, equal numbers per model, strided over each "
                                           "model's batch")
    return out


def main() -> int:
    if len(sys.argv) in (7, 8) and sys.argv[1] == "--summarize-rocprof":
        return summarize_rocprof(*sys.argv[2:])
    if len(sys.argv) >= 4 and sys.argv[1] == "--summarize-trace":
        return summarize_trace(*sys.argv[2:])
    if len(sys.argv) >= 4 and sys.argv[1] == "--summarize-counters":
        return summarize_counters(*sys.argv[2:])
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="grid72", choices=["grid72", "plane288", "mixed", "c1"])
    ap.add_argument("--precision", default="auto", choices=["auto", "fp64", "fp32", "mixed"],
                    help="grid72 only; the other workloads run FP64")
    ap.add_argument("--schedule", default="rounds", choices=["rounds", "persistent", "both"],
                    help="grid72: decimation schedule for Ndim <= 80 (both: time persistent over "
                         "a few steps, then rounds in full)")
    ap.add_argument("--nk", type=int, default=None,
                    help="k points (grid72: on the path, default 512; plane288: per side, default 257)")
    ap.add_argument("--nomega", type=int, default=None, help="grid72 energies (default 512)")
    ap.add_argument("--cpu-workers", type=int, default=None,
                    help="CPU baseline processes (default: one per usable core, capped by "
                         "OMP_NUM_THREADS when set)")
    ap.add_argument("--cpu-per-worker", type=int, default=None,
                    help="CPU baseline solves per worker (default 1200 grid72, 18 plane288, "
                         "60 per model mixed, 80000 c1: 10-20 s of CPU work each)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--plane-nw", type=int, default=PLANE_NW,
                    help="plane288 orbitals (default 144, Ndim 288; up to 192, Ndim 384)")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MIB",
                    help="only run a plain device copy of MIB MiB (counter calibration)")
    args = ap.parse_args()
    if args.cpu_workers is None:
        args.cpu_workers = default_cpu_workers()

    if args.calibrate_copy:
        import torch
        n = args.calibrate_copy * (1 << 20) // 4
        x = torch.ones(n, dtype=torch.float32, device="cuda:0")
        y = torch.empty_like(x)
        torch.cuda.synchronize()
        y.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": 4 * n, "copy_bytes_written": 4 * n}), flush=True)
        return 0

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU only: the surface Green's function path is not "
              "sharded across GPUs in this build (run with --gpus 1)", file=sys.stderr)
        return 2

    from wannier_tools_amd.surface import SurfaceGF

    run = {"grid72": run_grid72, "plane288": run_plane288, "mixed": run_mixed,
           "c1": run_c1}[args.workload]
    out = run(args, SurfaceGF)
    if "cpu_baseline" in out:
        log(f"[bench] cpu: {out['cpu_baseline']['value']:.1f} solves/s")
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
