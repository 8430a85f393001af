"""Benchmark: 2-site DMRG sweeps/s at chi = 1024 on one MI355X.

Workload (one "step" = one full 2-site DMRG sweep, 2(N-1) = 198 region steps):
  spin-1/2 XXZ chain, Delta = 1, N = 100, open boundaries, MPO bond dim 5, d = 2;
  seeded random initial MPS (bond dim 8, i.i.d. N(0,1), normalised);
  maxdim ramp 64 -> 256 -> 1024 -> 1024 during the untimed warm-up sweeps,
  cutoff 1e-12, Lanczos krylovdim 3, maxiter 1; timed sweeps at maxdim 1024.
The timed form runs the H_eff contractions in --precision (default fp32 MFMA)
with FP64 Lanczos, environments and factorisation; one further FP64-plain sweep
from the same state gives the FP64 throughput and the energy difference
|dE/E| between the forms (both energies are FP64 <psi|H|psi>).

Prints ONE JSON line (see the repository's bench contract).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_TFLOPS = {"fp64": 78.6, "fp32": 157.3, "bf16x3": 2500.0, "bf16": 2500.0}
HBM_PEAK_GBS = 8000.0


# Single-kernel classes timed live in the timed sweeps (HIP events carried by the
# launches themselves, on the context stream): the roofline is reported for the one
# with the largest summed time.  name -> (kernel, bound, unit of the peak)
ROOF_CLASSES = {
    "fact_reduce": "k_bidiag / k_sytrd (one-launch bidiagonalisation / tridiagonalisation of factorize)",
    "heff_gemm1": "k_gemm_mfma H_eff GEMM1 (L . theta)",
    "heff_gemm2": "k_gemm_mfma H_eff GEMM2 (T3 . R^T, split-K reduction included)",
}
PROFILE_EVERY = 7    # launches per HIP-event sample and class in the timed sweeps (prime, so the
                     # sample walks through the positions of the launches within a region)


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--workload", default="chain", choices=["chain", "qn", "tree-tdvp", "readme"],
                   help="chain: dense XXZ N=100 DMRG (the headline); qn: U(1) spin-1 N=64 block-sparse DMRG; "
                        "tree-tdvp: 2-site TDVP quench of the TFIM on a 63-site binary tree; readme: the "
                        "reference's README timing workload (spin-1 Heisenberg N=100, 5 sweeps, four forms)")
    p.add_argument("--steps", type=int, default=None,
                   help="timed sweeps (chain, qn: default 3) or time steps (tree-tdvp: default 20)")
    p.add_argument("--warmup", type=int, default=None,
                   help="untimed ramp sweeps (chain, qn: default 8; tree-tdvp: 0)")
    p.add_argument("--calibrate-copy", action="store_true",
                   help="run one 256 MiB device-to-device tensor copy first (counter calibration under rocprofv3)")
    p.add_argument("--precision", default="fp32", choices=["fp64", "fp32", "bf16x3", "bf16"])
    p.add_argument("--nsites", type=int, default=100)
    p.add_argument("--maxdim", type=int, default=None, help="chain, qn: 1024; tree-tdvp: 256")
    p.add_argument("--delta", type=float, default=1.0)
    p.add_argument("--cutoff", type=float, default=None, help="chain: 1e-12; qn, tree-tdvp: 1e-10")
    p.add_argument("--seed", type=int, default=0)
    p.add_argument("--no-fp64-plain", action="store_true", help="skip the FP64-plain comparison sweep")
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--cpu-seconds", type=float, default=20.0, help="budget of the CPU baseline sample")
    p.add_argument("--chi1024-steps", type=int, default=3,
                   help="chain: timed sweeps per form of the leg with every interior bond pinned at maxdim 1024 "
                        "(cutoff 0); 0 skips the leg")
    p.add_argument("--chi1024-forms", default="fp64,fp32,bf16x3",
                   help="chain: forms timed in the chi=1024 leg (comma separated; the first is the reference form)")
    p.add_argument("--serving-requests", type=int, default=40,
                   help="Poisson-stream requests of the serving leg (0 skips it)")
    p.add_argument("--serving-slots", type=int, default=8)
    a = p.parse_args()
    tree = a.workload == "tree-tdvp"
    if a.steps is None:
        a.steps = 20 if tree else 3
    if a.warmup is None:
        a.warmup = 0 if tree else 8
    if a.maxdim is None:
        a.maxdim = 256 if tree else 1024
    if a.cutoff is None:
        a.cutoff = 1e-12 if a.workload == "chain" else 1e-10
    return a


def ramp(maxdim, warmup):
    sched = [m for m in (64, 256, 1024) if m < maxdim] + [maxdim]
    while len(sched) < warmup:
        sched.append(maxdim)
    return sched[:warmup] if warmup > 0 else []


def run_sweeps(prob, nsweeps, maxdim, cutoff, precision, drain=None):
    """Continues the same problem (state and cached environments) for nsweeps.
    ``drain``: a context whose profile records are folded into its per-class
    totals after every sweep (bounds the number of live HIP events)."""
    from networksolvers_amd.sweep import eigsolve_problem
    nlog = len(prob.region_log)
    t_last = [time.perf_counter()]

    def progress(region_iter, *, sweep, nsweeps, **kw):
        now = time.perf_counter()
        p = region_iter.problem
        if drain is not None:
            drain.profile_stats()
        print(f"bench:   sweep {sweep}/{nsweeps} ({precision}) {now - t_last[0]:.2f} s  E={p.eigenvalue:.12f}  "
              f"maxlinkdim={p.state.maxlinkdim()}", file=sys.stderr, flush=True)
        t_last[0] = now

    E, psi = eigsolve_problem(prob, nsweeps=nsweeps, nsites=2, updater_kwargs=dict(precision=precision),
                              inserter_kwargs=dict(trunc=dict(cutoff=cutoff, maxdim=maxdim)),
                              sweep_printer=progress)
    return E, psi, prob.region_log[nlog:]


def gpu_sweeps(args):
    import networksolvers_amd as ns
    from networksolvers_amd import models
    ctx = ns.Context(0)
    if args.calibrate_copy:
        import numpy as np
        big = ctx.empty((1 << 25,), np.float64)        # 256 MiB
        big.copy().free()
        ctx.sync()
        big.free()
    N = args.nsites
    H = ns.TTNO(ctx, models.xxz_mpo(N, Jz=args.delta))
    psi = ns.TTN.from_arrays(ctx, models.random_mps(N, 2, 8, seed=args.seed))
    prob = ns.EigsolveProblem(state=psi, operator=ns.ProjTTN(H))
    sched = ramp(args.maxdim, args.warmup)
    t0 = time.perf_counter()
    if sched:
        run_sweeps(prob, len(sched), sched, args.cutoff, args.precision)
    ctx.sync()
    t_warm = time.perf_counter() - t0
    print(f"bench: warm-up {len(sched)} sweeps {sched} in {t_warm:.1f} s, maxlinkdim {prob.state.maxlinkdim()}",
          file=sys.stderr, flush=True)
    linkdims_start = prob.state.linkdims()
    # timed sweeps: HIP events carried by the H_eff GEMM launches themselves (on
    # the context stream), one launch in PROFILE_EVERY per class, for the roofline
    # of the dominant kernel; sampling keeps the event overhead out of the timing
    ctx.profile_classes(list(ROOF_CLASSES))
    ctx.profile_sampling(PROFILE_EVERY)
    ctx.profile(True)
    ctx.profile_reset()
    ctx.sync()
    w0 = time.monotonic_ns()
    t0 = time.perf_counter()
    E_ritz, psi, log = run_sweeps(prob, args.steps, args.maxdim, args.cutoff, args.precision)
    ctx.sync()
    t_timed = time.perf_counter() - t0
    print(f"bench: timed window monotonic_ns {w0} {time.monotonic_ns()}", file=sys.stderr, flush=True)
    stats = ctx.profile_stats()
    ctx.profile(False)
    ctx.profile_classes(None)
    ctx.profile_sampling(1)
    E_mixed = ns.expect_mpo(psi, H)
    print(f"bench: {args.steps} timed sweeps ({args.precision}) in {t_timed:.2f} s, E={E_mixed:.14f}",
          file=sys.stderr, flush=True)
    out = {"t_timed": t_timed, "E_mixed": E_mixed, "E_ritz": E_ritz, "stats": stats,
           "linkdims_start": linkdims_start, "linkdims_end": psi.linkdims(), "regions": len(log),
           "mps_host": psi.to_arrays() if not args.no_cpu_baseline else None,
           "kept_mean": sum(r[2] for r in log) / max(len(log), 1)}
    # one more sweep of the same form with events around every profiled launch:
    # the time shares come from it (events on every launch slow the host loop)
    ctx.profile(True)
    ctx.profile_reset()
    ctx.sync()
    t0 = time.perf_counter()
    run_sweeps(prob, 1, args.maxdim, args.cutoff, args.precision)
    ctx.sync()
    out["t_profiled"] = time.perf_counter() - t0
    out["stats_all"] = ctx.profile_stats()
    ctx.profile(False)
    if not args.no_fp64_plain and args.precision != "fp64":
        ctx.sync()
        t0 = time.perf_counter()
        _, psi64, _ = run_sweeps(prob, 1, args.maxdim, args.cutoff, "fp64")
        ctx.sync()
        out["t_fp64_sweep"] = time.perf_counter() - t0
        out["E_fp64"] = ns.expect_mpo(psi64, H)
        print(f"bench: 1 FP64-plain sweep in {out['t_fp64_sweep']:.2f} s, E={out['E_fp64']:.14f}",
              file=sys.stderr, flush=True)
    ctx.close()
    return out


CHI1024_RAMP = [64, 256, 1024, 1024]


def chi1024_leg(args):
    """The chain at its design point: XXZ Delta=1, N=100, seeded chi=8 random
    start, cutoff 0 so that maxdim binds, untimed sweeps on the ramp
    64, 256, 1024, 1024 (from there every bond i with 2^min(i, N-i) >= 1024 has
    dimension 1024, i.e. 81 of the 99 bonds; Gram matrices 2048 x 2048), then for
    each form ``chi1024_steps`` timed sweeps, every form starting from the same
    state (a device copy of the ramp's result, fresh environments).  Per form:
    sweeps/s, the FP64 <psi|H|psi> after its sweeps and |dE/E| against the first
    form's (FP64 plain); per-class kernel time shares and the H_eff GEMM roofline
    from HIP events on every launch of the timed sweeps (at these sizes an event
    costs microseconds against region steps of tens of milliseconds)."""
    import networksolvers_amd as ns
    from networksolvers_amd import models
    ctx = ns.Context(0)
    N = args.nsites
    H = ns.TTNO(ctx, models.xxz_mpo(N, Jz=args.delta))
    prob = ns.EigsolveProblem(state=ns.TTN.from_arrays(ctx, models.random_mps(N, 2, 8, seed=args.seed)),
                              operator=ns.ProjTTN(H))
    t0 = time.perf_counter()
    run_sweeps(prob, len(CHI1024_RAMP), CHI1024_RAMP, 0.0, "fp64")
    ctx.sync()
    start = prob.state
    dims = start.linkdims()
    print(f"bench: chi1024 ramp {CHI1024_RAMP} in {time.perf_counter() - t0:.1f} s, bonds at 1024: "
          f"{sum(1 for x in dims if x == 1024)} of {len(dims)}", file=sys.stderr, flush=True)
    forms = [f for f in args.chi1024_forms.split(",") if f]
    out = {"workload": f"2-site DMRG, XXZ Delta={args.delta} chain N={N}, maxdim 1024, cutoff 0 (maxdim binds), "
                       f"Lanczos K=3; untimed ramp {CHI1024_RAMP} from a seeded chi=8 start; every form starts "
                       f"from the ramp's state",
           "maxlinkdim_timed": max(dims), "bonds_at_1024": sum(1 for x in dims if x == 1024),
           "steps": args.chi1024_steps, "forms": {}}
    ref_E = None
    for form in forms:
        p = ns.EigsolveProblem(state=start.copy(), operator=ns.ProjTTN(H))
        ctx.profile_classes(None)
        ctx.profile_sampling(1)
        ctx.profile(True)
        ctx.profile_reset()
        ctx.sync()
        t0 = time.perf_counter()
        _, psi, log = run_sweeps(p, args.chi1024_steps, 1024, 0.0, form, drain=ctx)
        ctx.sync()
        dt = time.perf_counter() - t0
        stats = ctx.profile_stats()
        ctx.profile(False)
        E = ns.expect_mpo(psi, H)
        if ref_E is None:
            ref_E = E
        prof_ms = sum(v["total_ms"] for v in stats.values())
        share = {k: round(v["total_ms"] / (1e3 * dt), 4) for k, v in stats.items() if v["launches"]}
        peak = PEAK_TFLOPS[form]
        roof = {}
        for cls in ("heff_gemm1", "heff_gemm2"):
            st = stats[cls]
            if st["total_ms"] > 0:
                tf = st["flops"] / (st["total_ms"] * 1e-3) / 1e12
                roof[cls] = {"achieved_tflops": round(tf, 2), "peak": peak, "frac": round(tf / peak, 4),
                             "avg_ms": round(st["total_ms"] / st["launches"], 4), "launches": st["launches"]}
                if form == "bf16x3":
                    # the matrix cores issue three bf16 products (hi.hi, hi.lo, lo.hi) per
                    # algorithmic product: their utilisation is three times frac
                    roof[cls]["mfma_products"] = 3
                    roof[cls]["mfma_frac"] = round(3 * tf / peak, 4)
        dom = max((k for k in stats if stats[k]["launches"]), key=lambda k: stats[k]["total_ms"])
        out["forms"][form] = {"sweeps_per_s": round(args.chi1024_steps / dt, 5), "s_per_sweep": round(dt / max(args.chi1024_steps, 1), 3),
                              "E": E, "rel_dE_vs_" + forms[0]: abs(E - ref_E) / abs(ref_E),
                              "mean_kept": round(sum(r[2] for r in log) / max(len(log), 1), 1),
                              "time_share": share, "kernel_time_share_total": round(prof_ms / (1e3 * dt), 4),
                              "dominant_class": dom, "heff_roofline": roof}
        print(f"bench: chi1024 {form}: {args.chi1024_steps} sweeps in {dt:.2f} s, E={E:.14f}, dominant {dom} "
              f"({share.get(dom)})", file=sys.stderr, flush=True)
        del p, psi
    base = out["forms"][forms[0]]["sweeps_per_s"]
    for form in forms:
        out["forms"][form]["speedup_vs_" + forms[0]] = round(out["forms"][form]["sweeps_per_s"] / base, 3)
    ctx.close()
    return out


def cpu_baseline(args, budget_s, mps_host):
    """The oracle (numpy/OpenBLAS FP64 restatement of the region loop) on a
    bounded sample of the same workload: region steps of the next sweep, started
    from the converged state the GPU run reached (downloaded to the host), run
    until the budget is spent.  The first region (which also pays for the gauge
    walk and for building every environment) is excluded; sweeps/s = 1 / (198 x
    mean region time)."""
    from oracle import chain, models
    W = models.xxz_mpo(args.nsites, Jz=args.delta)
    res = chain.dmrg_chain(W, mps_host, nsweeps=1, maxdim=args.maxdim, cutoff=args.cutoff,
                           max_seconds=budget_s)
    times = [r.seconds for r in res.log[1:]] or [res.log[0].seconds]
    t_region = sum(times) / len(times)
    nreg = 2 * (args.nsites - 1)
    try:
        threads = int(os.environ.get("OMP_NUM_THREADS") or os.environ.get("OPENBLAS_NUM_THREADS") or 0)
    except ValueError:
        threads = 0
    if threads <= 0:
        threads = len(os.sched_getaffinity(0))
    mean_kept = sum(r.kept for r in res.log) / len(res.log)
    return {"value": 1.0 / (nreg * t_region), "unit": "sweeps/s", "cores": threads, "kind": "port",
            "sample": f"{len(times)} region steps (of {nreg} per sweep) of the next 2-site sweep from the converged "
                      f"chi<={max(a.shape[2] for a in mps_host)} state (mean kept {mean_kept:.0f}), "
                      f"{1e3 * t_region:.1f} ms each, numpy/OpenBLAS FP64 restatement; first region excluded"}


def serving_leg(args):
    """The mixed-size serving stream (XXZ chains N ~ U{16..128}, Delta ~ U[0,2],
    maxdim ~ U{64,128,256}, 4 sweeps, cutoff 1e-10, FP32 H_eff form): saturated
    throughput from a burst queued at t=0, then a Poisson stream at 0.8x that
    rate for p50/p99 latency; a few requests are re-solved in FP64 for the
    energy error of the form."""
    import networksolvers_amd as ns
    from networksolvers_amd import serving
    srv = serving.Server(slots=args.serving_slots)
    try:
        burst = serving.make_stream(max(2 * args.serving_slots, 8), rate=0.0, seed=args.seed + 1)
        res_b, wall_b = srv.run(burst, realtime=False)
        sat = len([r for r in res_b if r.error is None]) / wall_b
        rate = 0.8 * sat
        stream = serving.make_stream(args.serving_requests, rate=rate, seed=args.seed + 2)
        print(f"[bench] serving: saturated {sat:.2f} solves/s; stream of {len(stream)} at {rate:.2f}/s",
              file=sys.stderr, flush=True)
        def progress(done, total, secs):
            print(f"[bench] serving: {done}/{total} requests done in {secs:.1f} s", file=sys.stderr, flush=True)
        res, wall = srv.run(stream, realtime=True, progress=progress, progress_every=max(10, len(stream) // 20))
    finally:
        srv.close()
    ok = [r for r in res if r.error is None]
    lat = serving.latency_stats(res)
    # FP64 re-solve of a few requests: energy error of the FP32 form
    ctx = ns.Context(0)
    errs = []
    try:
        for r in ok[:4]:
            req = stream[r.rid]
            req64 = serving.SolveRequest(**{**req.__dict__, "precision": "fp64"})
            e64, _, _ = serving.run_solve(ctx, req64)
            errs.append(abs(r.energy - e64) / abs(e64))
    finally:
        ctx.close()
    return {"workload": "XXZ chains N~U{16..128}, Delta~U[0,2], maxdim~U{64,128,256}, 4 sweeps, cutoff 1e-10, "
                        "fp32 H_eff + f64 Krylov/factorize",
            "requests": len(stream), "completed": len(ok), "slots": args.serving_slots,
            "saturated_solves_per_s": round(sat, 3), "arrival_rate_per_s": round(rate, 3),
            "solves_per_s": round(len(ok) / wall, 3), "p50_latency_s": lat["p50_s"], "p99_latency_s": lat["p99_s"],
            "mean_latency_s": lat["mean_s"], "max_rel_dE_vs_fp64": max(errs) if errs else None,
            "peak_concurrency": srv.peak_concurrency}


def _traffic_from_profile(cls):
    """HBM bytes per launch of the roofline kernel from the committed counter summary of
    the same workload (two rocprofv3 --pmc runs, FETCH_SIZE and WRITE_SIZE, scaled by
    what the counters read for a device copy of known size); None when there is none."""
    path = os.path.join(ROOT, "profiles", f"{cls}_traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        t = json.load(f)
    return {"bytes_per_launch": t["hbm_bytes_per_launch"], "source": f"profiles/{cls}_traffic.json ({t['how']})"}


def _common(args, metric, value, unit, total_ms, steps, dtype, config, roofline, share):
    return {"metric": metric, "value": round(value, 6), "unit": unit, "n_gpus": 1, "steps": steps,
            "warmup": args.warmup, "ms_per_step": round(total_ms / max(steps, 1), 3), "higher_is_better": True,
            "scaling": "weak", "vs_baseline": None, "dtype": dtype, "data": "synthetic", "config": config,
            "roofline": roofline, "time_share": share}


def _roofline(stats, cls, total_ms, peak=PEAK_TFLOPS["fp64"]):
    s = stats[cls]
    achieved = s["flops"] / (s["total_ms"] * 1e-3) / 1e12 if s["total_ms"] > 0 else 0.0
    share = {k: round(v["total_ms"] / total_ms, 4) for k, v in stats.items() if v["launches"]}
    return ({"bound": "mfma", "kernel": cls, "achieved": round(achieved, 3), "peak": peak, "unit": "TFLOP/s",
             "frac": round(achieved / peak, 4), "traffic": None, "launches": s["launches"],
             "avg_ms": round(s["total_ms"] / max(s["launches"], 1), 4),
             "flops_per_launch": s["flops"] / max(s["launches"], 1)}, share)


def qn_workload(args):
    """Block-sparse U(1) DMRG: spin-1 Heisenberg chain N=64, MPO D=5, total Sz=0
    from a Neel product state grown by the densitymatrix subspace expansion
    (expansion factor 1.5, in every sweep; it stops adding vectors once a link
    reaches maxdim); untimed 2-site sweeps on the maxdim ramp 32, 64, 128, 256,
    512, then maxdim, then the timed sweeps at maxdim (H_eff block programs in
    --precision, environments, expansion and factorisation FP64, Lanczos K=3);
    one further FP64-plain sweep from the same state gives the FP64 throughput and
    |dE/E| between the forms (FP64 <psi|H|psi>)."""
    import networksolvers_amd as ns
    from networksolvers_amd import models, qn
    from networksolvers_amd.sweep import eigsolve_problem
    ctx = ns.Context(0)
    N = 64
    site = qn.spin_site_index(3)
    H = qn.QNMPO(ctx, models.heisenberg_mpo(N, d=3), site)
    states = [2 if i % 2 == 0 else 0 for i in range(N)]
    prob = ns.EigsolveProblem(state=qn.qn_product_mps(ctx, states, site), operator=ns.sweep.projected_operator(H))
    sched = ([m for m in (32, 64, 128, 256, 512) if m < args.maxdim] + [args.maxdim] * args.warmup)[:args.warmup]

    if args.precision not in ("fp64", "fp32"):
        raise SystemExit("qn serves --precision fp64 or fp32")

    def sweeps(n, maxdim, precision=args.precision):
        t = [time.perf_counter()]

        def progress(region_iter, *, sweep, nsweeps, **kw):
            p = region_iter.problem
            now = time.perf_counter()
            print(f"bench:   qn sweep {sweep}/{nsweeps} {now - t[0]:.2f} s  E={p.eigenvalue:.12f}  "
                  f"maxlinkdim={p.state.maxlinkdim()}", file=sys.stderr, flush=True)
            t[0] = now
        trunc = dict(cutoff=args.cutoff, maxdim=maxdim)
        return eigsolve_problem(prob, nsweeps=n, nsites=2, sweep_printer=progress,
                                extracter_kwargs=dict(trunc=trunc, subspace_algorithm="densitymatrix"),
                                updater_kwargs=dict(precision=precision), inserter_kwargs=dict(trunc=trunc))

    if sched:
        sweeps(len(sched), sched)
    ctx.sync()
    w0 = time.monotonic_ns()
    t0 = time.perf_counter()
    E, psi = sweeps(args.steps, args.maxdim)
    ctx.sync()
    t_timed = time.perf_counter() - t0
    print(f"bench: timed window monotonic_ns {w0} {time.monotonic_ns()}", file=sys.stderr, flush=True)
    nsec = max(len(psi.links[i]) for i in range(N + 1))
    E_psi = ns.expect_mpo(psi, H)
    # one more sweep with per-launch HIP events for the roofline and time shares
    ctx.profile(True)
    ctx.profile_reset()
    t0 = time.perf_counter()
    sweeps(1, args.maxdim)
    ctx.sync()
    t_prof = time.perf_counter() - t0
    stats = ctx.profile_stats()
    ctx.profile(False)
    table = ctx.tune_table()
    tuner = {"classes": len(table), "decided": sum(r["choice"] != -1 for r in table),
             "chose_64": sum(r["choice"] == 64 for r in table)}
    plain = None
    if args.precision != "fp64":
        ctx.sync()
        t0 = time.perf_counter()
        _, psi64 = sweeps(1, args.maxdim, "fp64")
        ctx.sync()
        t64 = time.perf_counter() - t0
        E64 = ns.expect_mpo(psi64, H)
        plain = {"sweeps_per_s": round(1.0 / t64, 6), "speedup_of_form": round(t64 * args.steps / t_timed, 3),
                 "E_fp64_after_sweep": E64, "rel_dE": abs(E_psi - E64) / abs(E64)}
    ctx.close()
    total_ms = 1e3 * t_timed
    roof, share = _roofline(stats, "block", 1e3 * t_prof, PEAK_TFLOPS[args.precision])
    config = {"workload": f"2-site U(1) block-sparse DMRG, spin-1 Heisenberg chain N={N}, d=3, MPO D=5, total Sz=0 "
                          f"(Neel start, densitymatrix subspace expansion), maxdim {args.maxdim}, "
                          f"cutoff {args.cutoff:g}, Lanczos K=3",
              "precision": args.precision, "regions_per_sweep": 2 * (N - 1), "maxlinkdim_timed": psi.maxlinkdim(),
              "max_sectors_per_link": nsec, "energy": E_psi, "parallelism": "single GPU"}
    line = _common(args, "QN DMRG sweeps/s (spin-1 N=64, Sz=0)", args.steps / t_timed, "sweeps/s", total_ms,
                   args.steps, {"fp64": "f64", "fp32": "f32+f64"}[args.precision], config, roof, share)
    if plain:
        line["fp64_plain"] = plain
    line["block_gemm_tiles"] = tuner
    return line


# The reference's own wall times for this workload (README.md:169-181, the
# optimal_map code state; hardware unstated; Julia @time of the whole dmrg call).
README_SECONDS = {"2site_dense": 5.8, "2site_qn": 5.5, "1site_dense_expand": 9.8, "1site_qn_expand": 7.7}


def readme_workload(args):
    """The reference's README timing workload (examples/timed_dmrg/timed_dmrg.jl,
    README.md:119-181): spin-1 Heisenberg chain N=100 from the Neel state ("Up" on
    even sites), 5 sweeps, cutoff 1e-9, maxdim [10, 40, 80, 160], in four forms:
    2-site dense, 2-site U(1) QN, and 1-site with the densitymatrix expansion
    (max_expand 4) dense and QN.  Each form runs once untimed for one sweep (library
    start-up), then the whole 5-sweep solve from a fresh product state is timed,
    environments included, as the reference's @time is.  FP64 plain (the
    reference's arithmetic); the line's value is the 2-site dense wall time."""
    import networksolvers_amd as ns
    from networksolvers_amd import models, qn
    from networksolvers_amd.sweep import eigsolve_problem
    ctx = ns.Context(0)
    N, d = 100, 3
    W = models.heisenberg_mpo(N, d=d)
    states = [0 if (i + 1) % 2 == 0 else 2 for i in range(N)]      # "Up" (m=+1) on even 1-based sites
    maxdim, cutoff, nsw = [10, 40, 80, 160], 1e-9, 5
    trunc = dict(cutoff=cutoff, maxdim=maxdim)
    site = qn.spin_site_index(d)
    H_dense = ns.TTNO(ctx, W)
    H_qn = qn.QNMPO(ctx, W, site)

    def problem(form):
        if "qn" in form:
            return ns.EigsolveProblem(state=qn.qn_product_mps(ctx, states, site),
                                      operator=ns.sweep.projected_operator(H_qn))
        return ns.EigsolveProblem(state=ns.TTN.from_arrays(ctx, models.product_mps(states, d)),
                                  operator=ns.ProjTTN(H_dense))

    def solve(form, nsweeps):
        nsites = 1 if form.startswith("1site") else 2
        ek = dict(trunc=trunc)
        if "expand" in form:
            ek.update(subspace_algorithm="densitymatrix", max_expand=4)
        prob = problem(form)
        return eigsolve_problem(prob, nsweeps=nsweeps, nsites=nsites, extracter_kwargs=ek,
                                inserter_kwargs=dict(trunc=trunc))

    forms = ["2site_dense", "2site_qn", "1site_dense_expand", "1site_qn_expand"]
    res = {}
    for form in forms:
        solve(form, 1)
        ctx.sync()
        t0 = time.perf_counter()
        E, psi = solve(form, nsw)
        ctx.sync()
        dt = time.perf_counter() - t0
        res[form] = {"seconds": round(dt, 4), "energy": E, "maxlinkdim": psi.maxlinkdim(),
                     "reference_seconds": README_SECONDS[form],
                     "speedup_vs_reference": round(README_SECONDS[form] / dt, 3)}
        print(f"bench: readme {form}: {dt:.3f} s for {nsw} sweeps, E={E:.12f}, maxlinkdim={psi.maxlinkdim()} "
              f"(reference {README_SECONDS[form]} s)", file=sys.stderr, flush=True)
    ctx.close()
    v = res["2site_dense"]["seconds"]
    line = _common(args, "DMRG wall time, spin-1 Heisenberg N=100, 5 sweeps (README timing workload)", v, "s",
                   1e3 * v, nsw, "f64", {"workload": "S=1 Heisenberg chain N=100, Neel start, cutoff 1e-9, maxdim "
                                                     "[10,40,80,160], 5 sweeps; 2-site dense timed as the value",
                                         "parallelism": "single GPU"}, None, None)
    line.update(higher_is_better=False, vs_baseline=round(v / README_SECONDS["2site_dense"], 4), forms=res,
                warmup=1)
    return line


def tree_tdvp_workload(args):
    """2-site TDVP quench, order 4, exponentiate solver: H = -sum ZZ - h sum X
    (h = 1) on the complete binary tree of 63 sites, all-up start, dt = 0.05;
    the timed steps are the first ``steps`` time steps (default 20, t = 1).  The
    timed form is --precision (ComplexF32 MFMA contraction programs with FP64
    Krylov exponentiate for fp32); the ComplexF64-plain form is timed the same
    way, and the fidelity and <Z_v> profile of the form are reported against it."""
    import numpy as np
    import networksolvers_amd as ns
    from networksolvers_amd import tree as ptree
    if args.precision not in ("fp64", "fp32"):
        raise SystemExit("tree-tdvp serves --precision fp64 or fp32")
    ctx = ns.Context(0)
    n = 63
    V = list(range(n))
    G = ns.Graph(V, [((i - 1) // 2, i) for i in range(1, n)])
    H = ns.TreeTTNO(ctx, G, ns.tfim_tree_mpo(G, h=1.0))
    psi0 = ns.product_ttn(ctx, G, {v: 0 for v in V}, 2)
    dt = 0.05
    times = [dt * k for k in range(args.warmup + args.steps + 1)]
    Z = np.diag([1.0, -1.0])
    leaves = [v for v in V if 2 * v + 1 >= n]

    def run(precision, window=False):
        marks, wmarks = [], []

        def progress(region_iter, *, sweep, nsweeps, **kw):
            ctx.sync()
            marks.append(time.perf_counter())
            wmarks.append(time.monotonic_ns())
            print(f"bench:   tdvp ({precision}) step {sweep}/{nsweeps} t={dt * sweep:.2f}  "
                  f"maxlinkdim={region_iter.problem.state.maxlinkdim()}", file=sys.stderr, flush=True)
        kws = dict(nsites=2, tdvp_order=4, updater_kwargs=dict(solver=ns.exponentiate_solver, precision=precision),
                   inserter_kwargs=dict(trunc=dict(cutoff=args.cutoff, maxdim=args.maxdim)))
        w0 = time.monotonic_ns()
        t0 = time.perf_counter()
        psi = ns.tdvp(H, psi0, times, sweep_printer=progress, **kws)
        ctx.sync()
        t_end = time.perf_counter()
        t_start = marks[args.warmup - 1] if args.warmup > 0 else t0
        if window:
            w_start = wmarks[args.warmup - 1] if args.warmup > 0 else w0
            print(f"bench: timed window monotonic_ns {w_start} {time.monotonic_ns()}", file=sys.stderr, flush=True)
        return psi, t_end - t_start, kws

    psi, t_timed, kws = run(args.precision, window=True)
    z = ns.expect_local(psi, Z)
    plain = None
    if args.precision != "fp64":
        psi64, t64, _ = run("fp64")
        z64 = ns.expect_local(psi64, Z)
        ov = ptree.inner(psi64, psi)
        fid = abs(ov) ** 2 / abs(ptree.inner(psi64, psi64) * ptree.inner(psi, psi))
        plain = {"steps_per_s": round(args.steps / t64, 6), "speedup_of_form": round(t64 / t_timed, 3),
                 "fidelity_vs_fp64": fid, "max_abs_dZ_vs_fp64": max(abs(z[v] - z64[v]) for v in V),
                 "maxlinkdim_end_fp64": psi64.maxlinkdim()}
    # one more time step from the final state with per-launch HIP events (roofline, time shares)
    ctx.profile(True)
    ctx.profile_reset()
    t0 = time.perf_counter()
    ns.tdvp(H, psi, [0.0, dt], sweep_printer=lambda *a, **k: None, **kws)
    ctx.sync()
    t_prof = time.perf_counter() - t0
    stats = ctx.profile_stats()
    ctx.profile(False)
    ctx.close()
    total_ms = 1e3 * t_timed
    peak = PEAK_TFLOPS[args.precision]
    roof, share = _roofline(stats, "net", 1e3 * t_prof, peak)
    config = {"workload": f"2-site TDVP (order 4, Krylov exponentiate) quench of H=-sum ZZ - 1.0 sum X on the "
                          f"complete binary tree of {n} sites, all-up start, dt {dt}, maxdim {args.maxdim}, "
                          f"cutoff {args.cutoff:g}",
              "precision": args.precision, "regions_per_step": 6 * (2 * (n - 1) - 1), "time": dt * args.steps,
              "maxlinkdim_end": psi.maxlinkdim(),
              "Z_root": float(np.real(z[0])), "Z_leaves_mean": float(np.mean([np.real(z[v]) for v in leaves])),
              "parallelism": "single GPU"}
    line = _common(args, "TDVP time steps/s (63-site binary-tree TFIM, 2-site, order 4)", args.steps / t_timed,
                   "steps/s", total_ms, args.steps, {"fp64": "c128", "fp32": "c64+c128"}[args.precision], config,
                   roof, share)
    if plain:
        line["complex128_plain"] = plain
    return line


def summarize_rocprof(root, window_log=None, top=25):
    """Text summary of a rocprofv3 output folder (-f csv): the --stats table, the
    dispatches inside the bench's timed window (bounds printed to stderr as
    "timed window monotonic_ns A B"; rocprofv3 timestamps share that clock), and
    per-kernel means of PMC counters.  Prints the summary."""
    import collections
    import csv
    import glob
    window = None
    if window_log and os.path.exists(window_log):
        for line in open(window_log):
            if "timed window monotonic_ns" in line:
                a, b = line.split()[-2:]
                window = (int(a), int(b))
    out = []
    for f in glob.glob(os.path.join(root, "**", "*kernel_stats.csv"), recursive=True):
        rows = sorted(csv.DictReader(open(f)), key=lambda r: -float(r.get("TotalDurationNs", 0) or 0))
        out.append(f"== {os.path.basename(f)} (all dispatches of the command, top {top} by total time)")
        if rows:
            out.append(",".join(rows[0].keys()))
        out += [",".join(str(v) for v in r.values()) for r in rows[:top]]
    for f in glob.glob(os.path.join(root, "**", "*kernel_trace.csv"), recursive=True):
        agg = collections.defaultdict(lambda: [0, 0])
        spans = []
        n = 0
        for r in csv.DictReader(open(f)):
            n += 1
            st, en = int(r["Start_Timestamp"]), int(r["End_Timestamp"])
            if window and window[0] <= st <= window[1]:
                a = agg[r.get("Kernel_Name", "?")]
                a[0] += 1
                a[1] += en - st
                spans.append((st, min(en, window[1])))
        out.append(f"== {os.path.basename(f)}: {n} dispatches; timed window {window}")
        if spans:
            # device-busy time: the union of the dispatch intervals inside the window
            spans.sort()
            busy, cur_s, cur_e = 0, spans[0][0], spans[0][1]
            for a, b in spans[1:]:
                if a > cur_e:
                    busy += cur_e - cur_s
                    cur_s, cur_e = a, b
                else:
                    cur_e = max(cur_e, b)
            busy += cur_e - cur_s
            length = window[1] - window[0]
            out.append(f"-- window {length / 1e6:.3f} ms, {len(spans)} dispatches, device busy {busy / 1e6:.3f} ms "
                       f"({busy / length:.3f} of the window: union of the dispatch intervals)")
        if agg:
            out.append("-- dispatches inside the timed window (name, calls, total_ms, avg_us)")
            for name, (c, t) in sorted(agg.items(), key=lambda kv: -kv[1][1])[:top]:
                out.append(f"{name[:150]}, {c}, {t / 1e6:.3f}, {t / c / 1e3:.3f}")
            out.append("-- every MFMA GEMM and split-K reduction inside the timed window (name, calls, total_ms, avg_us)")
            for name, (c, t) in sorted(agg.items(), key=lambda kv: -kv[1][1]):
                if "k_gemm_mfma" in name or "k_splitk_reduce" in name:
                    out.append(f"{name[:150]}, {c}, {t / 1e6:.3f}, {t / c / 1e3:.3f}")
    for f in glob.glob(os.path.join(root, "**", "*counter_collection.csv"), recursive=True):
        agg = collections.defaultdict(lambda: [0, 0.0, 0.0])
        aggw = collections.defaultdict(lambda: [0, 0.0])
        for r in csv.DictReader(open(f)):
            key = (r.get("Kernel_Name", "?"), r.get("Counter_Name", "?"))
            a = agg[key]
            v = float(r.get("Counter_Value", 0) or 0)
            a[0] += 1
            a[1] += v
            a[2] = max(a[2], v)
            st = int(r.get("Start_Timestamp", 0) or 0)
            if window and window[0] <= st <= window[1]:
                aggw[key][0] += 1
                aggw[key][1] += v
        out.append(f"== {os.path.basename(f)}")
        out.append("-- kernel, counter, dispatches, mean value per dispatch, largest value of one dispatch")
        for (k, c), (nn, sm, mx) in sorted(agg.items(), key=lambda kv: -kv[1][1]):
            out.append(f"{k[:150]}, {c}, {nn}, {sm / nn:.1f}, {mx:.1f}")
        if aggw:
            out.append(f"-- dispatches inside the timed window {window} (kernel, counter, dispatches, mean value)")
            for (k, c), (nn, sm) in sorted(aggw.items(), key=lambda kv: -kv[1][1]):
                out.append(f"{k[:150]}, {c}, {nn}, {sm / nn:.1f}")
    for f in glob.glob(os.path.join(root, "**", "*results.db"), recursive=True):
        out += _summarize_rocpd(f, window, top)
    print("\n".join(out), flush=True)


def _summarize_rocpd(path, window, top):
    """The same summary from rocprofv3's SQLite output (its default format): every
    dispatch of the command by total time, the dispatches inside the timed window, and
    per-kernel means of collected counters."""
    import collections
    import sqlite3
    con = sqlite3.connect(path)
    out = []
    rows = con.execute("select name, start, end from kernels").fetchall()
    agg = collections.defaultdict(lambda: [0, 0])
    aggw = collections.defaultdict(lambda: [0, 0])
    for name, st, en in rows:
        agg[name][0] += 1
        agg[name][1] += en - st
        if window and window[0] <= st <= window[1]:
            aggw[name][0] += 1
            aggw[name][1] += en - st
    tot = sum(t for _, t in agg.values())
    out.append(f"== {os.path.basename(path)}: {len(rows)} dispatches, {tot / 1e6:.3f} ms of kernel time")
    out.append("-- all dispatches (name, calls, total_ms, avg_us, share)")
    for name, (cn, t) in sorted(agg.items(), key=lambda kv: -kv[1][1])[:top]:
        out.append(f"{name[:150]}, {cn}, {t / 1e6:.3f}, {t / cn / 1e3:.3f}, {t / max(tot, 1):.4f}")
    if aggw:
        totw = sum(t for _, t in aggw.values())
        out.append(f"-- dispatches inside the timed window {window}: {totw / 1e6:.3f} ms of kernel time "
                   f"in {(window[1] - window[0]) / 1e6:.3f} ms (name, calls, total_ms, avg_us, share of kernel time)")
        for name, (cn, t) in sorted(aggw.items(), key=lambda kv: -kv[1][1])[:top]:
            out.append(f"{name[:150]}, {cn}, {t / 1e6:.3f}, {t / cn / 1e3:.3f}, {t / max(totw, 1):.4f}")
    try:
        pmc = con.execute("select * from counters_collection").fetchall()
        cols = [d[0] for d in con.execute("select * from counters_collection").description]
    except sqlite3.Error:
        pmc, cols = [], []
    if pmc:
        ki = cols.index("kernel_name") if "kernel_name" in cols else cols.index("name")
        ci = cols.index("counter_name")
        vi = cols.index("value") if "value" in cols else cols.index("counter_value")
        si = cols.index("start") if "start" in cols else None
        pagg = collections.defaultdict(lambda: [0, 0.0])
        paggw = collections.defaultdict(lambda: [0, 0.0])
        for r in pmc:
            key = (r[ki], r[ci])
            pagg[key][0] += 1
            pagg[key][1] += float(r[vi] or 0)
            if window and si is not None and window[0] <= int(r[si] or 0) <= window[1]:
                paggw[key][0] += 1
                paggw[key][1] += float(r[vi] or 0)
        out.append("-- counters (kernel, counter, dispatches, mean value per dispatch)")
        for (k, cn), (n, sm) in sorted(pagg.items(), key=lambda kv: -kv[1][1])[:3 * top]:
            out.append(f"{k[:150]}, {cn}, {n}, {sm / n:.1f}")
        if paggw:
            out.append(f"-- counters inside the timed window {window}")
            for (k, cn), (n, sm) in sorted(paggw.items(), key=lambda kv: -kv[1][1])[:3 * top]:
                out.append(f"{k[:150]}, {cn}, {n}, {sm / n:.1f}")
    return out


def main():
    if len(sys.argv) > 2 and sys.argv[1] == "--summarize-rocprof":
        summarize_rocprof(sys.argv[2], sys.argv[3] if len(sys.argv) > 3 else None)
        return
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; --gpus above 1 is not served (the sweep "
                                   "would shard by MPO channel or real space; see the design notes)"}))
        sys.exit(2)
    if args.workload != "chain":
        line = {"qn": qn_workload, "tree-tdvp": tree_tdvp_workload, "readme": readme_workload}[args.workload](args)
        print(json.dumps(line), flush=True)
        return
    r = gpu_sweeps(args)
    value = args.steps / r["t_timed"]
    st = r["stats"]
    # dominant kernel: the single-kernel class with the largest summed time in the timed sweeps
    dom = max(ROOF_CLASSES, key=lambda k: st[k]["total_ms"])
    s = st[dom]
    achieved = s["flops"] / (s["total_ms"] * 1e-3) / 1e12 if s["total_ms"] > 0 else 0.0
    # the reductions run FP64 vector arithmetic whatever the H_eff form
    peak = PEAK_TFLOPS["fp64"] if dom == "fact_reduce" else PEAK_TFLOPS[args.precision]
    total_ms = 1e3 * r["t_timed"]
    prof_ms = 1e3 * r["t_profiled"]
    share = {k: round(v["total_ms"] / prof_ms, 4) for k, v in r["stats_all"].items() if v["launches"]}
    gemm = max(("heff_gemm1", "heff_gemm2"), key=lambda k: st[k]["total_ms"])
    sg = st[gemm]
    gach = sg["flops"] / (sg["total_ms"] * 1e-3) / 1e12 if sg["total_ms"] > 0 else 0.0
    gpeak = PEAK_TFLOPS[args.precision]
    traffic = _traffic_from_profile(dom)
    line = {
        "metric": "DMRG sweeps/s at chi=1024 (MFMA vs FP64 plain, dE<=1e-9); p50/p99 solve latency",
        "value": round(value, 6),
        "unit": "sweeps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(total_ms / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp64": "f64", "fp32": "f32", "bf16x3": "bf16x3", "bf16": "bf16"}[args.precision] + "+f64",
        "data": "synthetic",
        "config": {"workload": f"2-site DMRG, XXZ Delta={args.delta} chain N={args.nsites}, d=2, MPO D=5, "
                               f"maxdim {args.maxdim}, cutoff {args.cutoff:g}, Lanczos K=3",
                   "precision": args.precision, "regions_per_sweep": 2 * (args.nsites - 1),
                   "maxlinkdim_timed": max(r["linkdims_start"]), "mean_kept": round(r["kept_mean"], 1),
                   "parallelism": "single GPU"},
        "roofline": {"bound": "mfma", "kernel": ROOF_CLASSES[dom], "class": dom, "achieved": round(achieved, 5),
                     "peak": peak, "unit": "TFLOP/s", "frac": round(achieved / peak, 6),
                     "traffic": traffic["bytes_per_launch"] if traffic else None,
                     "traffic_source": traffic["source"] if traffic else None,
                     "launches": s["launches"], "sampled_one_in": PROFILE_EVERY,
                     "avg_ms": round(s["total_ms"] / max(s["launches"], 1), 4),
                     "flops_per_launch": s["flops"] / max(s["launches"], 1),
                     "algorithmic_bytes_per_launch": s["bytes"] / max(s["launches"], 1)},
        "roofline_heff_gemm": {"bound": "mfma", "kernel": ROOF_CLASSES[gemm], "class": gemm,
                               "achieved": round(gach, 3), "peak": gpeak, "unit": "TFLOP/s",
                               "frac": round(gach / gpeak, 4), "launches": sg["launches"],
                               "avg_ms": round(sg["total_ms"] / max(sg["launches"], 1), 4),
                               "flops_per_launch": sg["flops"] / max(sg["launches"], 1)},
        "time_share": share,
        "time_share_sweep_s": round(r["t_profiled"], 3),
        "energy": {"E_form": r["E_mixed"], "E_ritz_last_region": r["E_ritz"]},
    }
    if "t_fp64_sweep" in r:
        line["fp64_plain"] = {"sweeps_per_s": round(1.0 / r["t_fp64_sweep"], 6),
                              "speedup_of_form": round(value * r["t_fp64_sweep"], 3),
                              "E_fp64_after_sweep": r["E_fp64"],
                              "rel_dE": abs(r["E_mixed"] - r["E_fp64"]) / abs(r["E_fp64"])}
    if args.chi1024_steps > 0:
        line["chi1024"] = chi1024_leg(args)
    if args.serving_requests > 0:
        line["serving"] = serving_leg(args)
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(args, args.cpu_seconds, r["mps_host"])
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
