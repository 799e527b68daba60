#!/usr/bin/env python
"""FM-DBZP search throughput on one MI355X.

One step = one `acquire_` over the benchmark workload: GPS L1 C/A, 16.368 MHz
real int16 IF samples at 4.092 MHz, 80 ms = 8 noncoherent segments of 10 ms
coherent integration, PRNs 1..32 searched (8 present, CN0 30-40 dB-Hz, 50 bps
data), Doppler +-7 kHz (160 bins of 100 Hz), bit-edge search over 10
alignments. The samples are resident in HBM before the timed region; the
plan (code FFTs, tables, workspace) is built beforehand, as the reference's
benchmarks do (benchmark/benchmarks.jl:120-124).

Prints ONE JSON line. value = search cells/s = sum over PRNs of
get_num_cells (ndop x spc x R) per step / wall time per step.
"""
import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "acquisition.jl_amd"))

METRIC = "search cells/s + PRN acqs/s on 1 GPU, mixed-prec vs FP32 at equal peak bins"
HBM_PEAK_GBS = 8000.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def hbm_stream(nbytes: int):
    """Copy, read-only and write-only streams of libhbmcopy.so over `nbytes`:
    the HBM bandwidth this device reaches in practice (the roofline peak stays
    the 8 TB/s datasheet figure)."""
    import ctypes
    lib = ctypes.CDLL(os.path.join(ROOT, "acquisition.jl_amd", "acquisition", "_lib", "libhbmcopy.so"))
    lib.hbm_stream_run.argtypes = [ctypes.c_size_t, ctypes.c_int, ctypes.c_int]
    lib.hbm_stream_run.restype = ctypes.c_double
    out = {"bytes": nbytes}
    for kind, name, moved in ((0, "copy", 2), (1, "read", 1), (2, "write", 1)):
        ms = lib.hbm_stream_run(nbytes, 10, kind)
        if ms <= 0:
            raise SystemExit(f"hbm stream {name} failed ({ms})")
        out[f"{name}_gb_per_s"] = round(moved * nbytes / (ms * 1e-3) / 1e9, 1)
    print(json.dumps(out), flush=True)


def copy_calibration(nbytes: int):
    """Time the plain copy kernel of libhbmcopy.so. Profiled with the
    FETCH_SIZE / WRITE_SIZE counters, its per-dispatch readings over
    `nbytes` are the scale factors for the engine kernels' readings."""
    import ctypes
    lib = ctypes.CDLL(os.path.join(ROOT, "acquisition.jl_amd", "acquisition", "_lib", "libhbmcopy.so"))
    lib.hbm_copy_run.argtypes = [ctypes.c_size_t, ctypes.c_int]
    lib.hbm_copy_run.restype = ctypes.c_double
    ms = lib.hbm_copy_run(nbytes, 5)
    if ms <= 0:
        raise SystemExit(f"copy calibration failed ({ms})")
    print(json.dumps({"copy_bytes": nbytes, "read_kib": nbytes / 1024, "write_kib": nbytes / 1024,
                      "ms_per_copy": round(ms, 4), "gb_per_s": round(2 * nbytes / (ms * 1e-3) / 1e9, 1)}),
          flush=True)


KERNEL_CLASS_OF = {"k_corr_tile": "corr_tile", "k_column_simple": "column", "k_column_sign": "column",
                   "k_column_rotation": "column", "k_column_c160": "column", "k_column_c160_pair": "column",
                   "k_column_rot2000": "column", "k_column_rot25": "column", "k_column_bitsplit": "column",
                   "k_column_reg": "column",
                   "k_full_corr": "column", "k_full31_corr": "column",
                   "k_column_rotsplit": "column", "k_corr_fc": "corr_tile", "k_fc_signal": "signal_fft",
                   "k_fc_code": "code_fft", "k_full_code": "code_fft", "k_full31_code": "code_fft",
                   "k_full_fold": "signal_fft", "k_full_signal": "signal_fft", "k_full31_signal": "signal_fft",
                   "k_signal_fft": "signal_fft", "k_reduce_rows": "reduce", "k_reduce_cols": "reduce",
                   "k_merge_rows": "reduce", "k_finalize": "finalize", "k_code_fft": "code_fft",
                   "k_export": "export", "k_export_cm": "export", "k_export_chip": "export",
                   "k_column_rotbig": "column", "k_column_rotmma": "column", "k_reduce_chunk": "reduce",
                   "k_colsum_chunk": "reduce", "k_merge_rows_nbr": "reduce", "k_finalize_chunked": "finalize"}
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "hbm_traffic_l1ca_16mhz_32prn.json")


def _cpu_model() -> str:
    """The host CPU's model name and logical core count (Linux)."""
    try:
        with open("/proc/cpuinfo") as f:
            names = [l.split(":", 1)[1].strip() for l in f if l.startswith("model name")]
        return f"{names[0]} ({len(names)} logical cores)" if names else "unknown"
    except OSError:
        return "unknown"


def pmc_summary(base: str, config_key: str):
    """Per-dispatch HBM bytes of each engine kernel class from four rocprofv3
    --pmc CSV outputs under `base` (pmc_fetch, pmc_write: this workload;
    pmc_copy_fetch, pmc_copy_write: the plain copy of --copy-calibration),
    each counter scaled by copied bytes / counter reading of the copy kernel."""
    import csv

    def per_dispatch(name, counter):
        sums, counts = {}, {}
        with open(os.path.join(base, name, "run_counter_collection.csv")) as f:
            for r in csv.DictReader(f):
                if r["Counter_Name"] != counter:
                    continue
                k = r["Kernel_Name"].split("(")[0].split("<")[0].replace("void ", "").strip()
                sums[k] = sums.get(k, 0.0) + float(r["Counter_Value"])
                counts[k] = counts.get(k, 0) + 1
        return {k: sums[k] / counts[k] for k in sums}

    cf, cw = per_dispatch("pmc_copy_fetch", "FETCH_SIZE"), per_dispatch("pmc_copy_write", "WRITE_SIZE")
    copy_kib = 1024.0 * 1024.0  # --copy-calibration 1024 (MiB)
    fs, ws = copy_kib / cf["hbm_copy_calibration"], copy_kib / cw["hbm_copy_calibration"]
    f, w = per_dispatch("pmc_fetch", "FETCH_SIZE"), per_dispatch("pmc_write", "WRITE_SIZE")
    out = {"config_key": config_key, "fetch_scale": round(fs, 4), "write_scale": round(ws, 4), "kernels": {}}
    # a class served by several kernels (the column-major reduction is two
    # passes) sums its kernels' per-dispatch bytes
    for k in f:
        cls = KERNEL_CLASS_OF.get(k)
        if cls and k in w:
            e = out["kernels"].setdefault(cls, {"kernel": "", "fetch_kib": 0.0, "write_kib": 0.0, "hbm_bytes": 0})
            e["kernel"] = (e["kernel"] + " + " + k) if e["kernel"] else k
            e["fetch_kib"] = round(e["fetch_kib"] + f[k], 1)
            e["write_kib"] = round(e["write_kib"] + w[k], 1)
            e["hbm_bytes"] += int(f[k] * fs * 1024 + w[k] * ws * 1024)
    print(json.dumps(out, indent=1))


def measured_traffic(kernel_class: str, config_key: str):
    """HBM bytes per launch of `kernel_class` recorded by pmc_summary for this
    workload configuration, or None when no matching record exists."""
    try:
        with open(TRAFFIC_FILE) as f:
            rec = json.load(f)
    except (OSError, ValueError):
        return None
    if rec.get("config_key") != config_key:
        return None
    k = rec.get("kernels", {}).get(kernel_class)
    return k["hbm_bytes"] if k else None


def _workspace_estimate(plan_host, nprn: int, budget: float) -> float:
    """Device bytes a plan of this geometry takes: signal-FFT cache plus the
    PRN-batch tile and accumulator, the batch limited by the per-plan budget
    (searches accumulated in code-column chunks take about the budget)."""
    nb, ndop, F = plan_host.num_blocks, plan_host.num_doppler_bins, plan_host.fft_size
    tp = (plan_host.block_size + 31) // 32 * 32
    ap_ = (plan_host.samples_per_code_eff + 31) // 32 * 32
    per_prn = nb * ndop * tp * 8 + ndop * ap_ * 4
    batch = max(1, min(nprn, int(budget // per_prn)))
    return min(batch * per_prn, budget) + plan_host.num_noncoherent_accumulations * ndop * F * 8


def _request_cells(r, h):
    return len(r.prns) * h.num_doppler_bins * h.samples_per_code * h.num_secondary_rotations


C5_WORKSPACE_GB = 24.0  # per plan; the code-column chunk width of the E1-like searches follows it
C5_GROUP_GB = 200.0     # plans of one submission, together


def _c5_groups(reqs, hosts, nsteps):
    """The batch in seeded order, cut into `nsteps` consecutive groups of as
    equal a request count as possible."""
    n = len(reqs)
    nsteps = max(1, min(nsteps, n))
    bounds = [round(i * n / nsteps) for i in range(nsteps + 1)]
    return [list(zip(reqs[bounds[i]:bounds[i + 1]], hosts[bounds[i]:bounds[i + 1]])) for i in range(nsteps)]


def _run_c5_group(grp, precision, timing):
    """Build the group's plans (one per geometry), generate its samples on the
    device, then time one `acquire_batch` submission of the whole group, in
    sub-submissions when the plans would not fit device memory together.
    Returns (seconds, results per request, kernel times per plan geometry)."""
    from acquisition import acquire_batch, plan_acquire
    from acquisition._native import ELTYPE

    budget = C5_WORKSPACE_GB * 2**30
    subs, cur, cur_b = [], [], 0.0
    for r, h in grp:
        est = _workspace_estimate(h, len(r.prns), budget)
        if cur and cur_b + est > C5_GROUP_GB * 2**30:
            subs.append(cur)
            cur, cur_b = [], 0.0
        cur.append((r, h))
        cur_b += est
    if cur:
        subs.append(cur)
    tot, results, ktimes = 0.0, [], {}
    for sub in subs:
        union = {}
        for r, h in sub:
            union.setdefault(r.plan_key(), (r, set()))[1].update(r.prns)
        plans = {}
        sigs = []
        try:
            for k, (r, ps) in union.items():
                plans[k] = plan_acquire(r.system, r.sampling_freq, sorted(ps), min_doppler_coverage=r.coverage,
                                        num_coherently_integrated_code_periods=r.num_coh,
                                        num_noncoherent_accumulations=r.num_nc,
                                        tile_precision=precision)
                if timing:
                    plans[k].native.set_timing(True)
            sigs = [r.signal(device=True) for r, h in sub]
            batch = [(plans[r.plan_key()], s, r.prns, {"subsample_interpolation": True})
                     for (r, h), s in zip(sub, sigs)]
            t0 = time.perf_counter()
            res = acquire_batch(batch)
            tot += time.perf_counter() - t0
            results += res
            if timing:
                for k, pl in plans.items():
                    ktimes[k] = (pl, pl.native.kernel_times())
        finally:
            for s in sigs:
                s.free()
            for k, pl in plans.items():
                if k not in ktimes:
                    pl.close()
    for k, (pl, kt) in ktimes.items():
        ktimes[k] = ({"ndop": pl.num_doppler_bins, "spc": pl.samples_per_code, "nb": pl.num_blocks,
                      "bs": pl.block_size, "F": pl.fft_size, "R": pl.num_secondary_rotations,
                      "nnc": pl.num_noncoherent_accumulations,
                      "kernel": pl.native.call_kernels(ELTYPE["cf32"], 1).split()[-1]}, kt)
        pl.close()
    return tot, results, ktimes


def run_mixed_batch(args):
    """The batched uneven mix: 256 requests drawn by seed from three types with
    no caps (E1-like searches up to +-50 kHz, 36 PRNs and N_nc 8). The batch is
    cut into --steps consecutive groups; one step is one `acquire_batch`
    submission of one group (its plans built and its samples generated on the
    device before the timed region), so the timed steps cover the whole batch
    once. The first --warmup groups also run once, untimed, beforehand.
    value = sum of get_num_cells over all requests / sum of step times."""
    from collections import Counter, defaultdict
    from acquisition import is_detected
    from acquisition.plan import _plan_host
    from acquisition.signals import mixed_batch_requests

    os.environ["FMDBZP_WORKSPACE_GB"] = str(C5_WORKSPACE_GB)
    reqs = mixed_batch_requests(n=args.batch_requests)
    hosts = [_plan_host(r.system, r.sampling_freq, r.prns, min_doppler_coverage=r.coverage,
                        num_coherently_integrated_code_periods=r.num_coh, num_noncoherent_accumulations=r.num_nc)
             for r in reqs]
    groups = _c5_groups(reqs, hosts, args.steps)
    cells_all = sum(_request_cells(r, h) for r, h in zip(reqs, hosts))
    dwell_all = sum(_request_cells(r, h) * r.num_nc for r, h in zip(reqs, hosts))
    log(f"mixed batch: {len(reqs)} requests {dict(Counter(r.kind for r in reqs))}, {cells_all:.3e} cells, "
        f"{dwell_all:.3e} cell-dwells, {len(groups)} steps")
    for gi in range(min(args.warmup, len(groups))):
        dt, _, _ = _run_c5_group(groups[gi], "fp32", False)
        log(f"warmup step {gi + 1}/{args.warmup}: {len(groups[gi])} requests, {dt:.3f} s")

    legs = {}
    run_legs = ("fp32",) if args.no_mixed else {"both": ("fp32", "mixed"), "fp32": ("fp32",),
                                                 "mixed": ("mixed",)}[args.c5_legs]
    for leg in run_legs:
        prec = "fp32" if leg == "fp32" else "auto"
        tot, res_all, det, col_geo = 0.0, [], Counter(), defaultdict(lambda: [0.0, 0, 0.0, None])
        kern = defaultdict(float)
        for gi, grp in enumerate(groups):
            dt, res, kt = _run_c5_group(grp, prec, True)
            tot += dt
            res_all += res
            for geo, times in kt.values():
                for k, (ms, n) in times.items():
                    kern[k] += ms
                c = col_geo[tuple(sorted(geo.items()))]
                c[0] += times["column"][0]
                c[1] += times["column"][1]
                c[3] = geo
            log(f"{leg} step {gi + 1}/{len(groups)}: {len(grp)} requests "
                f"{dict(Counter(r.kind for r, h in grp))}, {dt:.3f} s")
        for (r, h), rr in zip([x for g in groups for x in g], res_all):
            for x in rr:
                key = "present" if x.prn in r.present else "absent"
                det[key] += 1
                det[key + "_detected"] += int(is_detected(x))
        legs[leg] = dict(t=tot, res=res_all, det=det, kern=dict(kern), col_geo=dict(col_geo))
        log(f"{leg}: {tot:.2f} s, {cells_all / tot:.4e} cells/s, detections {dict(det)}")

    def leg_roofline(lg):
        """Roofline of the leg's dominant kernel: the column stage of the
        geometry with the largest column time. Algorithmic bytes per launch:
        the coherent tile read and the accumulator read-modify-write (write
        only at a PRN's first step) of the cells it covers."""
        if not lg["col_geo"]:
            return None
        key, (ms, nl, _, geo) = max(lg["col_geo"].items(), key=lambda kv: kv[1][0])
        ndop, spc, R, nnc = geo["ndop"], geo["spc"], geo["R"], geo["nnc"]
        nprn_steps = sum(len(r.prns) * r.num_nc for (r, h) in zip(reqs, hosts)
                         if (h.num_doppler_bins, h.samples_per_code, h.num_secondary_rotations,
                             h.num_noncoherent_accumulations) == (ndop, spc, R, nnc))
        nprn_first = nprn_steps // max(nnc, 1)
        alg = (nprn_steps * 8 * ndop * spc + (nprn_steps - nprn_first) * 8 * ndop * spc * R
               + nprn_first * 4 * ndop * spc * R)
        avg = ms / nl
        bpl = alg / nl
        ach = bpl / (avg * 1e-3) / 1e9
        flops = nprn_steps * spc * R * 5.0 * ndop * math.log2(ndop)
        out = {"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
               "frac": round(ach / HBM_PEAK_GBS, 4), "traffic": None, "kernel": geo["kernel"],
               "geometry": {k: v for k, v in geo.items() if k != "kernel"}, "launches": nl,
               "avg_launch_ms": round(avg, 4), "algorithmic_bytes_per_launch": int(bpl),
               "fft_equiv_tflops": round(flops / (ms * 1e-3) / 1e12, 2)}
        if geo["kernel"].startswith("k_column_rotmma") and ndop % 625 == 0:
            # issued matrix-core work: per column and rotation, n1 groups of 8
            # 32x32x16 and 16 32x32x8 FP16 products (padded operands)
            mf = nprn_steps * spc * R * (ndop // 625) * (8 * 32768 + 16 * 16384)
            out["mfma_tflops"] = round(mf / (ms * 1e-3) / 1e12, 2)
            out["mfma_frac_of_2500"] = round(mf / (ms * 1e-3) / 1e12 / 2500.0, 4)
        return out

    fp = legs.get("fp32")
    roofline = leg_roofline(fp) if fp else None
    mixed = None
    if "mixed" in legs:
        mx = legs["mixed"]
        mixed = {"form": "per request: FP16-operand DFT-matrix products on the matrix cores for the E1-like "
                         "rotation searches at +-25 and +-50 kHz (n1 = 10, 20), else the FP32 path",
                 "value": round(cells_all / mx["t"], 1), "seconds": round(mx["t"], 3),
                 "kernel_seconds": {k: round(v / 1e3, 3) for k, v in mx["kern"].items() if v},
                 "detections": dict(mx["det"]), "roofline": leg_roofline(mx)}
        if fp:
            mixed["speedup_vs_fp32"] = round(fp["t"] / mx["t"], 3)
            mixed["detections_equal"] = all(is_detected(a) == is_detected(b)
                                            for ra, rb in zip(fp["res"], mx["res"]) for a, b in zip(ra, rb))
            mixed["peak_bins_equal_detected"] = all(
                (a.engine_stats["row"], a.engine_stats["col"]) == (b.engine_stats["row"], b.engine_stats["col"])
                for ra, rb in zip(fp["res"], mx["res"]) for a, b in zip(ra, rb) if is_detected(a))
    main = fp if fp else legs["mixed"]
    cpu = None
    if not args.no_cpu_baseline:
        sys.path.insert(0, os.path.join(ROOT, "oracle"))
        import oracle
        from acquisition.plan import plan_code_samples  # noqa: F401  (the oracle builds the codes)

        t_cpu, c_cpu, names = 0.0, 0, []
        for r, h in zip(reqs, hosts):
            if r.kind == "c" or t_cpu > 15.0:
                continue
            sig = r.signal(device=False)
            t0 = time.perf_counter()
            oracle.acquire(h, sig, list(range(len(r.prns))), nthreads=args.cpu_threads)
            t_cpu += time.perf_counter() - t0
            c_cpu += _request_cells(r, h)
            names.append(r.kind)
        if c_cpu:
            cpu = {"value": round(c_cpu / t_cpu, 1), "unit": "search cells/s", "cores": args.cpu_threads,
                   "kind": "port",
                   "sample": f"{len(names)} type a / b requests of the same batch ({dict(Counter(names))}), "
                             f"C restatement in FP32, {args.cpu_threads} OpenMP threads, {t_cpu:.1f} s; the E1-like "
                             "(type c) requests need over a minute of oracle time per PRN and step and are not sampled"}
            log(f"cpu baseline: {cpu['value']:.3e} cells/s over {len(names)} requests ({t_cpu:.1f}s)")
    out = {
        "metric": METRIC,
        "value": round(cells_all / main["t"], 1),
        "unit": "search cells/s",
        "n_gpus": 1,
        "steps": len(groups),
        "warmup": min(args.warmup, len(groups)),
        "ms_per_step": round(main["t"] * 1e3 / len(groups), 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": (f"batched mix of {len(reqs)} requests: GPS L1 C/A (5 / 16.368 MHz, N_coh 1-10, "
                                "1-32 PRNs), L5-like (30.69 MHz, N_coh 1 or 10, 10-chip secondary, 1-36 PRNs), "
                                "E1-like (25 MHz, N_coh 25, R 25, 1-36 PRNs); Doppler coverage +-5 to +-50 kHz, "
                                "N_nc 1-8, CN0 30-45 dB-Hz, complex baseband generated on the device; one step is "
                                f"one acquire_batch submission of 1/{len(groups)} of the batch"),
                   "requests_by_type": dict(Counter(r.kind for r in reqs)), "total_cells": cells_all,
                   "total_cell_dwells": dwell_all, "precision": "fp32" if fp else "auto",
                   "signal": "device-resident complex64",
                   "workspace_gb_per_plan": C5_WORKSPACE_GB},
        "prn_acqs_per_s": round(sum(len(x) for x in main["res"]) / main["t"], 2),
        "cell_dwells_per_s": round(dwell_all / main["t"], 1),
        "kernel_seconds": {k: round(v / 1e3, 3) for k, v in main["kern"].items() if v},
        "detections": dict(main["det"]),
        "mixed_precision": mixed,
        "roofline": roofline,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--edge-steps", type=int, default=10)
    ap.add_argument("--literal-edges", action="store_true",
                    help="evaluate every bit-edge offset (the default evaluates one: with one data bit per "
                         "coherent block the offsets are circular rotations of the column)")
    ap.add_argument("--workload", choices=("c2", "c1", "c3", "c4", "c5", "e1wide"), default="c2",
                    help="c2 (default): GPS L1 C/A 16.368 MHz int16 IF, 32 PRNs, N_coh 10, N_nc 8; "
                         "c1: GPS L1 C/A 5 MHz, 1 ms, 32 PRNs; c3: the c2 search on quantised complex samples "
                         "(--c3-kind); c4: E1-like 25 MHz, 36 PRNs, N_coh 25, R 25, N_nc 4; "
                         "c5: batched mix of uneven requests; e1wide: the mix's dominant geometry, E1-like "
                         "+-50 kHz, one present and one absent PRN (with --precision fp32 or mfma)")
    ap.add_argument("--c3-kind", choices=("ci8", "2bit"), default="ci8")
    ap.add_argument("--no-mixed", action="store_true", help="skip the mixed-precision leg")
    ap.add_argument("--main-only", action="store_true",
                    help="time the main leg alone, without the mixed, literal-edges and graph legs (counter runs)")
    ap.add_argument("--precision", choices=("fp32", "fp16", "mfma", "auto"), default="fp32",
                    help="single-plan workloads: the plan's tile_precision (value is then that form's rate)")
    ap.add_argument("--graph-leg", action="store_true",
                    help="also time the same calls on a graph-replay plan (always on for c1)")
    ap.add_argument("--c5-legs", choices=("both", "fp32", "mixed"), default="both",
                    help="c5: which precision legs to time (value is the FP32 leg's when it runs)")
    ap.add_argument("--batch-requests", type=int, default=256)
    ap.add_argument("--batch-group", type=int, default=16, help="c5: at most this many requests per submission")
    ap.add_argument("--batch-group-gb", type=float, default=120.0,
                    help="c5: at most this much plan workspace per submission")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-threads", type=int, default=16)
    ap.add_argument("--cpu-prns", type=int, default=16)
    ap.add_argument("--copy-calibration", type=float, default=0.0, metavar="MIB",
                    help="only run a plain device copy of MIB MiB (FETCH_SIZE/WRITE_SIZE counter calibration)")
    ap.add_argument("--pmc-summary", metavar="DIR",
                    help="only summarise rocprofv3 FETCH_SIZE/WRITE_SIZE CSV runs under DIR")
    ap.add_argument("--hbm-stream", type=float, default=0.0, metavar="MIB",
                    help="only measure copy / read / write streaming bandwidth over MIB MiB buffers")
    args = ap.parse_args()
    if args.main_only:
        args.no_mixed = True
    if args.hbm_stream > 0:
        hbm_stream(int(args.hbm_stream * 2**20))
        return
    if args.pmc_summary:
        pmc_summary(args.pmc_summary,
                    f"{args.workload}-E{args.edge_steps}-{'literal' if args.literal_edges else 'one-edge'}")
        return
    if args.copy_calibration > 0:
        copy_calibration(int(args.copy_calibration * 2**20))
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported "
              "(the engine runs on a single MI355X; across GPUs the search would shard by PRN and request)",
              file=sys.stderr)
        sys.exit(2)

    if args.workload == "c5":
        run_mixed_batch(args)
        return

    import numpy as np
    from acquisition import GPSL1CA, acquire_, is_detected, plan_acquire
    from acquisition.device import DeviceArray
    from acquisition.signals import l1ca_if_int16_scene

    t0 = time.time()
    if args.workload == "c2":
        sc = l1ca_if_int16_scene(seed=0x5EED0002)
        plan_kw = dict(num_coherently_integrated_code_periods=10, bit_edge_search_steps=args.edge_steps,
                       num_noncoherent_accumulations=8, min_doppler_coverage=7000.0,
                       literal_edges=args.literal_edges)
        workload = ("GPS L1 C/A 16.368 MHz real int16 at IF 4.092 MHz, 80 ms; PRNs 1-32 (8 present); "
                    f"N_coh 10, bit-edge steps {args.edge_steps}, N_nc 8, +-7 kHz")
    elif args.workload == "c3":
        from acquisition.signals import l1ca_quantized_scene
        sc = l1ca_quantized_scene(kind=args.c3_kind)
        plan_kw = dict(num_coherently_integrated_code_periods=10, bit_edge_search_steps=args.edge_steps,
                       num_noncoherent_accumulations=8, min_doppler_coverage=7000.0,
                       literal_edges=args.literal_edges)
        workload = ("GPS L1 C/A 16.368 MHz complex at IF 4.092 MHz, quantised to "
                    + ("Complex{Int8} (sigma 32 LSB)" if args.c3_kind == "ci8" else "2-bit {+-1, +-3} packed 4 per byte")
                    + f", 80 ms; PRNs 1-32 (8 present); N_coh 10, bit-edge steps {args.edge_steps}, N_nc 8, +-7 kHz")
    elif args.workload == "c1":
        from acquisition.signals import l1ca_5mhz_scene
        sc = l1ca_5mhz_scene()
        plan_kw = dict(min_doppler_coverage=7000.0)
        workload = "GPS L1 C/A 5 MHz complex baseband, 1 ms; PRNs 1-32 (1 present); N_coh 1, N_nc 1, +-7 kHz"
    elif args.workload == "e1wide":
        from acquisition.signals import e1like_scene
        sc = e1like_scene(seed=0x5EED0E02, n_periods=25, nnc=2, fs=25e6, nprn=8, npresent=2,
                          cn0_range=(34.0, 38.0))
        sc.prns = sorted(sc.present[:1] + [p for p in sc.prns if p not in sc.present][:1])
        plan_kw = dict(num_coherently_integrated_code_periods=25, num_noncoherent_accumulations=2,
                       min_doppler_coverage=50000.0)
        workload = ("E1-like pilots at 25 MHz, +-50 kHz (12500 Doppler bins), N_coh 25, R 25, N_nc 2, 2 x 100 ms; "
                    "one present and one absent PRN (the dominant geometry of the batched mix)")
    else:
        from acquisition.signals import e1like_scene
        sc = e1like_scene(n_periods=25, nnc=4, fs=25e6, nprn=36, npresent=6)
        plan_kw = dict(num_coherently_integrated_code_periods=25, num_noncoherent_accumulations=4,
                       min_doppler_coverage=7000.0)
        workload = ("E1-like pilots (4092-chip codes, BOC(1,1), 25-chip secondary) at 25 MHz, 4 x 100 ms; "
                    "PRNs 1-36 (6 present); N_coh 25, R 25, N_nc 4, +-7 kHz")
    nsamp = sc.signal.n if hasattr(sc.signal, "n") else sc.signal.shape[0]
    log(f"scene: {nsamp} samples, present {sc.present} ({time.time() - t0:.1f}s)")
    prns = list(sc.prns)
    if args.precision != "fp32":
        plan_kw = dict(plan_kw, tile_precision=args.precision)
    plan = plan_acquire(sc.system, sc.sampling_freq, prns, **plan_kw)
    from acquisition import Packed2BitSignal
    if isinstance(sc.signal, Packed2BitSignal):
        dev = Packed2BitSignal(DeviceArray(sc.signal.packed), sc.signal.n)
    else:
        dev = DeviceArray(sc.signal)
    ndop, spc, R = plan.num_doppler_bins, plan.samples_per_code, plan.num_secondary_rotations
    cells = len(prns) * ndop * spc * R
    log(f"plan: spc {spc} nb {plan.num_blocks} bs {plan.block_size} F {plan.fft_size} ndop {ndop} "
        f"path {plan.path} E {plan.bit_edge_search_steps} Nnc {plan.num_noncoherent_accumulations}")

    res = None
    for i in range(args.warmup):
        res = acquire_(plan, dev, prns, interm_freq=sc.interm_freq)
    if res is not None:
        log(f"warmup done; detected {sorted(r.prn for r in res if is_detected(r))} (present {sc.present})")

    # value: the steps without per-kernel events; then the same steps again with
    # HIP events around every launch for the per-kernel times (roofline)
    t0 = time.perf_counter()
    for i in range(args.steps):
        res = acquire_(plan, dev, prns, interm_freq=sc.interm_freq)
    t1 = time.perf_counter()
    dt = (t1 - t0) / args.steps
    det = sorted(r.prn for r in res if is_detected(r))
    plan.native.set_timing(True)
    t2 = time.perf_counter()
    for i in range(args.steps):
        acquire_(plan, dev, prns, interm_freq=sc.interm_freq)
    dt_ev = (time.perf_counter() - t2) / args.steps
    kt = plan.native.kernel_times()
    plan.native.set_timing(False)
    log(f"timed {args.steps} steps: {dt * 1e3:.3f} ms/step ({dt_ev * 1e3:.3f} with kernel events); kernel ms totals "
        + ", ".join(f"{k} {v[0]:.2f}/{v[1]}" for k, v in kt.items() if v[1]))

    # the same steps with the samples in host memory (pageable numpy array:
    # the library stages them through pinned memory and copies them over PCIe)
    t0 = time.perf_counter()
    for i in range(max(1, args.steps // 2)):
        acquire_(plan, sc.signal, prns, interm_freq=sc.interm_freq)
    dt_host = (time.perf_counter() - t0) / max(1, args.steps // 2)

    # roofline of the dominant kernel (algorithmic bytes per launch)
    F, nb = plan.fft_size, plan.num_blocks
    nnc = plan.num_noncoherent_accumulations
    spc_eff = plan.samples_per_code_eff
    launches_per_step = {k: v[1] / args.steps for k, v in kt.items()}
    batches = max(1, round(launches_per_step.get("corr_tile", 1) / nnc))
    nbat = len(prns) / batches
    # column: per PRN and call, every step's tile read once, the accumulator
    # written at the first pass and read and written at each later one (a
    # launch of k_column_c160_pair carries two steps: one pass per pair)
    col_launches = launches_per_step.get("column", 0)
    passes = col_launches / batches if col_launches else 1
    col_call = len(prns) * (nnc * 8 * ndop * spc + 4 * ndop * spc_eff + (passes - 1) * 8 * ndop * spc_eff)
    bytes_per_launch = {
        "corr_tile": nbat * (8 * F * ndop + 8 * F * nb + 8 * ndop * spc),
        "column": col_call / col_launches if col_launches else None,
        "signal_fft": nnc * plan.num_coherently_integrated_code_periods * spc * 2 + 8 * F * ndop * nnc,
        "reduce": nbat * 4 * ndop * spc_eff,
    }
    dom = max((k for k in kt if kt[k][1]), key=lambda k: kt[k][0])
    avg_ms = kt[dom][0] / kt[dom][1]
    bpl = bytes_per_launch.get(dom)
    if bpl and dom == "column" and plan.num_doppler_bins > 4000:
        # chunked accumulation (code-column windows): one call's column launches
        # cover each PRN-step's cells once between them. Per PRN-step, the tile
        # read (8 ndop spc) and the accumulator (spc_eff = spc R columns) read and
        # written, written only at the first step; mean over the steps
        acc = (8 * ndop * spc_eff * (nnc - 1) + 4 * ndop * spc_eff) / nnc
        bpl = len(prns) * nnc * (8 * ndop * spc + acc) / launches_per_step["column"]
    full = "corr_tile" not in launches_per_step or not kt["corr_tile"][1]
    roofline = None
    if full and dom == "column":
        # full-period correlation: one circular correlation of the code period
        # per PRN, Doppler row and step (product and inverse transform, 5 n log2 n
        # + 6 n float operations, power and sum 4 n), bound by the vector unit;
        # against the FP32 vector rate without packed instructions
        fl = len(prns) * nnc * ndop * spc * (5 * math.log2(spc) + 10) / launches_per_step["column"]
        tf = fl / (avg_ms * 1e-3) / 1e12
        roofline = {"bound": "fp32", "achieved": round(tf, 2), "peak": 78.6, "unit": "TFLOP/s",
                    "frac": round(tf / 78.6, 4), "traffic": None, "kernel": "full_corr",
                    "avg_launch_ms": round(avg_ms, 4), "algorithmic_flops_per_launch": int(fl),
                    "algorithmic_bytes_per_launch": int((8 + 4) * len(prns) * ndop * spc
                                                        / launches_per_step["column"])}
        bpl = None
    if bpl:
        ach = bpl / (avg_ms * 1e-3) / 1e9
        config_key = (f"{args.workload}-E{plan.bit_edge_search_steps}-"
                      f"{'literal' if args.literal_edges else 'one-edge'}")
        roofline = {"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                    "frac": round(ach / HBM_PEAK_GBS, 4), "traffic": measured_traffic(dom, config_key),
                    "kernel": dom,
                    "avg_launch_ms": round(avg_ms, 4), "algorithmic_bytes_per_launch": int(bpl)}
    # the same figures for every timed class with an algorithmic byte count
    # (at C2 the correlation and the column pairs take about equal time, so the
    # dominant class above can be either); with code-column chunks (ndop above
    # 4000) the per-launch formulas above hold for the dominant class only
    roofline_by_class = {}
    for k in () if full else ("corr_tile", "column"):
        b = bpl if k == dom else bytes_per_launch.get(k)
        if b and kt.get(k, (0, 0))[1] and not (plan.num_doppler_bins > 4000 and k != dom):
            ms = kt[k][0] / kt[k][1]
            a = b / (ms * 1e-3) / 1e9
            roofline_by_class[k] = {"achieved": round(a, 1), "frac": round(a / HBM_PEAK_GBS, 4),
                                    "avg_launch_ms": round(ms, 4), "algorithmic_bytes_per_launch": int(b),
                                    "launches_per_step": round(kt[k][1] / args.steps, 2)}
    kernel_share = {k: round(v[0] / args.steps, 4) for k, v in kt.items() if v[1]}

    # mixed-precision leg: the same search with the coherent tile in FP16
    mixed = None
    if args.workload in ("c2", "c3") and not args.no_mixed:
        plan16 = plan_acquire(sc.system, sc.sampling_freq, prns, tile_precision="fp16", **plan_kw)
        for i in range(args.warmup):
            res16 = acquire_(plan16, dev, prns, interm_freq=sc.interm_freq)
        t0 = time.perf_counter()
        for i in range(args.steps):
            res16 = acquire_(plan16, dev, prns, interm_freq=sc.interm_freq)
        dt16 = (time.perf_counter() - t0) / args.steps
        plan16.close()
        same_det = all(is_detected(a) == is_detected(b) for a, b in zip(res, res16))
        bins = [(a.engine_stats["row"], a.engine_stats["col"]) == (b.engine_stats["row"], b.engine_stats["col"])
                for a, b in zip(res, res16)]
        det_bins = all(e for e, a in zip(bins, res) if is_detected(a))
        mixed = {"form": "FP16 coherent tile under an exact power-of-two scale, FP32 arithmetic",
                 "value": round(cells / dt16, 1), "ms_per_step": round(dt16 * 1e3, 4),
                 "speedup_vs_fp32": round(dt / dt16, 3), "detections_equal": same_det,
                 "peak_bins_equal_detected": det_bins, "peak_bins_equal_all": f"{sum(bins)}/{len(bins)}",
                 "fp64_oracle_error": "tests/test_gpu_mixed.py: at most 1.8e-4 of the peak, 1.5e-3 per cell"}
        log(f"mixed (fp16 tile): {dt16 * 1e3:.3f} ms/step, x{dt / dt16:.3f}; detections equal {same_det}, "
            f"detected peak bins equal {det_bins}, all {sum(bins)}/{len(bins)}")

    # literal-edges leg: the same search evaluating every bit-edge offset as
    # the reference's loop does (src/noncoherent_integration.jl:670-685)
    literal = None
    if (args.workload in ("c2", "c3") and not args.literal_edges and plan.bit_edge_search_steps > 1
            and not args.main_only):
        kw_lit = dict(plan_kw, literal_edges=True)
        planl = plan_acquire(sc.system, sc.sampling_freq, prns, **kw_lit)
        for i in range(args.warmup):
            resl = acquire_(planl, dev, prns, interm_freq=sc.interm_freq)
        t0 = time.perf_counter()
        for i in range(args.steps):
            resl = acquire_(planl, dev, prns, interm_freq=sc.interm_freq)
        dtl = (time.perf_counter() - t0) / args.steps
        planl.close()
        literal = {"value": round(cells / dtl, 1), "ms_per_step": round(dtl * 1e3, 4),
                   "one_edge_speedup": round(dtl / dt, 3),
                   "detections_equal": all(is_detected(a) == is_detected(b) for a, b in zip(res, resl)),
                   "peak_bins_equal": all((a.engine_stats["row"], a.engine_stats["col"])
                                          == (b.engine_stats["row"], b.engine_stats["col"]) for a, b in zip(res, resl))}
        log(f"literal edges: {dtl * 1e3:.3f} ms/step ({literal['value']:.3e} cells/s)")

    # graph leg: the same calls on a plan that captures its launch sequence
    # once and replays it (FMDBZP_OPT_GRAPH); reported beside value
    graph = None
    if (args.graph_leg or args.workload == "c1") and not args.main_only:
        plang = plan_acquire(sc.system, sc.sampling_freq, prns, graphs=True, **plan_kw)
        for i in range(max(args.warmup, 2)):
            resg = acquire_(plang, dev, prns, interm_freq=sc.interm_freq)
        t0 = time.perf_counter()
        for i in range(args.steps):
            resg = acquire_(plang, dev, prns, interm_freq=sc.interm_freq)
        dtg = (time.perf_counter() - t0) / args.steps
        caps, reps = plang.native.graph_counts()
        plang.close()
        same = all(a.engine_stats == b.engine_stats and a.peak_to_noise_ratio == b.peak_to_noise_ratio
                   for a, b in zip(res, resg))
        graph = {"ms_per_step": round(dtg * 1e3, 4), "speedup_vs_eager": round(dt / dtg, 3),
                 "captures": caps, "replays": reps, "results_identical": same}
        log(f"graph replay: {dtg * 1e3:.4f} ms/step (eager {dt * 1e3:.4f}), {caps} captures, {reps} replays, "
            f"identical {same}")

    cpu = None
    if not args.no_cpu_baseline and args.workload not in ("c4", "e1wide"):
        sys.path.insert(0, os.path.join(ROOT, "oracle"))
        import oracle

        # like for like: the same edge evaluation as the GPU value (the one-edge
        # identity on the N_db = 1 sign path, or the literal loop with
        # --literal-edges), and the literal loop beside it
        one_edge = plan.path == 1 and plan.num_data_bits == 1 and plan.bit_edge_search_steps > 1
        like_one = one_edge and not args.literal_edges
        sub = list(range(min(args.cpu_prns * (2 if like_one else 1), len(prns))))
        t0 = time.perf_counter()
        oracle.acquire(plan, sc.signal, sub, if_hz=sc.interm_freq, nthreads=args.cpu_threads, one_edge=like_one)
        cdt = time.perf_counter() - t0
        cpu = {"value": round(len(sub) * ndop * spc * R / cdt, 1), "unit": "search cells/s",
               "cores": args.cpu_threads, "kind": "port", "cpu_model": _cpu_model(),
               "edge_evaluation": "one-edge identity" if like_one else "literal",
               "sample": f"PRNs 1..{len(sub)} of the same workload (all segments), C restatement in FP32, "
                         f"{args.cpu_threads} OpenMP threads over PRNs, "
                         f"{'one-edge identity' if like_one else 'literal edge loop'}, {cdt:.1f} s"}
        if like_one:
            sub2 = list(range(min(args.cpu_prns, len(prns))))
            t0 = time.perf_counter()
            oracle.acquire(plan, sc.signal, sub2, if_hz=sc.interm_freq, nthreads=args.cpu_threads)
            cdt2 = time.perf_counter() - t0
            cpu["literal_value"] = round(len(sub2) * ndop * spc * R / cdt2, 1)
            cpu["literal_sample"] = f"PRNs 1..{len(sub2)}, literal {plan.bit_edge_search_steps}-offset loop, {cdt2:.1f} s"
        log(f"cpu baseline: {cpu['value']:.3e} cells/s ({cdt:.1f}s)"
            + (f", literal edges {cpu['literal_value']:.3e}" if "literal_value" in cpu else ""))

    out = {
        "metric": METRIC,
        "value": round(cells / dt, 1),
        "unit": "search cells/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(dt * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32" if args.precision == "fp32" else "f16 operands, f32 accumulation",
        "data": "synthetic",
        "config": {"workload": workload,
                   "prns": len(prns), "samples_per_code": spc, "num_doppler_bins": ndop,
                   "num_blocks": nb, "fft_size": F, "num_coh": plan.num_coherently_integrated_code_periods,
                   "bit_edge_search_steps": plan.bit_edge_search_steps, "num_noncoherent": nnc,
                   "secondary_rotations": R, "precision": args.precision,
                   "signal": "device-resident " + ("packed 2-bit" if isinstance(sc.signal, Packed2BitSignal)
                                                    else str(sc.signal.dtype)),
                   "edge_evaluation": "literal" if args.literal_edges else "one-edge identity"},
        "prn_acqs_per_s": round(len(prns) / dt, 2),
        "host_signal_cells_per_s": round(cells / dt_host, 1),
        "cell_dwells_per_s": round(cells * nnc / dt, 1),
        "kernel_ms_per_step": kernel_share,
        "detected": det,
        "mixed_precision": mixed,
        "literal_edges_leg": literal,
        "graph_replay": graph,
        "roofline": roofline,
        "roofline_by_class": roofline_by_class,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)
    (dev.packed if isinstance(dev, Packed2BitSignal) else dev).free()
    plan.close()


if __name__ == "__main__":
    main()
