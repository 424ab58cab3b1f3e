"""Benchmark: transient instances/s of the batched ring-oscillator Monte Carlo
on one MI355X, next to the plain per-instance GPU path and the CPU oracle.

    python bench.py [--gpus 1] [--steps K] [--warmup W]

Workload (one "step" = one full batched transient over the whole batch):
  4096 ring oscillators, stage count N uniform odd in [11, 101] (uneven sizes,
  one launch), square-law inverters (NMOS Vth 0.4 V, KP 200 uA/V^2, W/L
  1u/0.18u; PMOS Vth -0.4 V, KP 80 uA/V^2, W/L 2u/0.18u), per-transistor Vth
  offset ~ N(0, 30 mV), 5 fF per stage, VDD 1.8 V, 0-10 ns from a seeded
  perturbed initial state, BDF2 at reltol 1e-6 / abstol 1e-9 V, FP64.

Inputs are uploaded before the timed region (they are resident in HBM when it
starts); the timed region is cs_batch_run (launch + completion).  The plain
per-instance path (host step control, one captured hipGraph launch per Newton
iteration) is timed on a sample of instances over the full 0-10 ns span, and
the CPU oracle (OpenMP across instances) on a bounded sample; both are
reported as instances/s.  Prints one JSON line.
"""
import argparse
import dataclasses
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "cedarsim.jl_amd"))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

HBM_PEAK = 8.0e12          # B/s, MI355X HBM3E
FP64_PEAK = 78.6e12        # FLOP/s, MI355X FP64 vector

PROFILES = os.path.join(ROOT, "profiles")


def measured(name, key):
    """A figure of a committed rocprofv3 summary (profiles/<name>.json), or
    None when the summary or the figure is absent."""
    try:
        with open(os.path.join(PROFILES, name + ".json")) as f:
            return json.load(f).get(key)
    except (OSError, ValueError):
        return None


def host_cpu():
    """(logical CPUs, model name) of the host, from /proc/cpuinfo."""
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return os.cpu_count() or 1, model


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--n-inst", type=int, default=4096)
    ap.add_argument("--t-stop", type=float, default=10e-9)
    ap.add_argument("--seed", type=int, default=2024)
    ap.add_argument("--plain-sample", type=int, default=1, help="instances timed on the plain path")
    ap.add_argument("--cpu-sample", type=int, default=0,
                    help="instances timed on the CPU oracle (0: four per thread, size-stratified)")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--adjoint-inst", type=int, default=1024,
                    help="also time the adjoint workload (51-stage rings, dE/dW, 0-5 ns) "
                         "with this many instances")
    ap.add_argument("--adjoint-only", action="store_true")
    ap.add_argument("--kernel", choices=["auto", "lds", "global"], default="auto",
                    help="batched kernel: LDS-resident plan (auto when it fits) or global plan")
    ap.add_argument("--bsim-inst", type=int, default=1 << 20,
                    help="BSIM-CMG device-eval microbenchmark size (0: skip)")
    ap.add_argument("--bsim-only", action="store_true")
    ap.add_argument("--grid-n", type=int, default=450,
                    help="power-grid workload: n x n RC mesh (0: skip)")
    ap.add_argument("--grid-inv", type=int, default=10_000, help="power-grid inverters")
    ap.add_argument("--grid-tstop", type=float, default=5e-9, help="power-grid transient span")
    ap.add_argument("--grid-only", action="store_true")
    ap.add_argument("--grid-newton", choices=["modified", "full"], default="modified",
                    help="power-grid transient: modified Newton (the step's first factorization reused by its "
                         "later iterations, as IDA does) or full Newton (refactor every iteration)")
    ap.add_argument("--copy-calib", type=int, default=0,
                    help="only fill and copy a buffer of this many MiB on the device (the known-size "
                         "kernels that scale the HBM byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; --gpus must be 1"}))
        sys.exit(2)

    if args.copy_calib:
        import torch
        nb = args.copy_calib << 20
        a = torch.empty(nb, dtype=torch.uint8, device="cuda:0")
        b = torch.empty_like(a)
        a.fill_(1)                  # a kernel that writes nb bytes
        tot = a.sum(dtype=torch.int64)   # a kernel that reads nb bytes
        b.copy_(a)                  # device copy (may run on a copy engine)
        torch.cuda.synchronize()
        print(json.dumps({"copy_calib_bytes": nb, "ok": bool(b[-1].item() == 1 and int(tot) == nb)}),
              flush=True)
        return

    import cedarhip as ch
    from cedarhip import lib as L
    from cedarhip.workloads import ring_mc, ring_widths

    if args.grid_only:
        eng = ch.Engine(0)
        print(json.dumps({"power_grid": grid_section(ch, L, args, eng)}), flush=True)
        eng.close()
        return
    if args.bsim_only:
        eng = ch.Engine(0)
        print(json.dumps({"device_eval": bsim_section(ch, args, eng)}), flush=True)
        eng.close()
        return
    if args.adjoint_only:
        eng = ch.Engine(0)
        print(json.dumps({"adjoint": adjoint_section(ch, L, ring_widths, args, eng)}), flush=True)
        eng.close()
        return

    log(f"building workload: {args.n_inst} rings, seed {args.seed}")
    flats, params, u0s, stages = ring_mc(n_inst=args.n_inst, seed=args.seed)
    kern = {"auto": L.BATCH_KERNEL_AUTO, "lds": L.BATCH_KERNEL_LDS,
            "global": L.BATCH_KERNEL_GLOBAL}[args.kernel]
    opts = ch.TranOptions(t_start=0.0, t_stop=args.t_stop, reltol=1e-6, abstol=1e-9,
                          init=L.INIT_UIC, max_order=2, n_out=0, dt_out=0.0, batch_kernel=kern)
    eng = ch.Engine(0)
    systems, key, inst_sys = [], {}, []
    for f in flats:
        if id(f) not in key:
            key[id(f)] = len(systems)
            systems.append(eng.load(f))
        inst_sys.append(key[id(f)])
    log(f"{len(systems)} distinct circuits compiled; uploading batch")
    batch = ch.Batch(eng, systems, inst_sys, params, opts, u0s)
    for w in range(args.warmup):
        ms = batch.run()
        log(f"warmup {w}: {ms:.1f} ms")
    times = []
    t0 = time.perf_counter()
    for k in range(args.steps):
        ms = batch.run()
        times.append(ms)
        log(f"step {k}: {ms:.1f} ms")
    wall = time.perf_counter() - t0
    res = batch.results(times[-1])
    bad = [i for i, s in enumerate(res.stats) if s.retcode != 0]
    if bad:
        log(f"{len(bad)} instances failed: first {bad[:5]} {[res.retcodes[i] for i in bad[:5]]}")
    ms_per_step = wall / args.steps * 1e3
    value = args.n_inst * args.steps / wall
    kernel_ms = float(np.mean(times))
    iters = sum(s.newton_iters for s in res.stats)
    steps_acc = sum(s.steps for s in res.stats)
    n_mos_tot = sum(len(systems[inst_sys[i]].flat.arrays["mos_vth"]) * res.stats[i].newton_iters
                    for i in range(args.n_inst))
    achieved = res.alg_bytes / (kernel_ms * 1e-3)
    out = {
        "metric": "transient instances/sec at reltol 1e-6, batched vs plain (1 GPU); device evals/s",
        "value": value,
        "unit": "instances/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {
            "workload": (f"ring-oscillator Monte Carlo: {args.n_inst} rings, N odd U[11,101], "
                         f"sigma_vth 30 mV, 5 fF/stage, VDD 1.8 V, 0-{args.t_stop * 1e9:g} ns, "
                         "BDF2 reltol 1e-6 abstol 1e-9 V"),
            "n_inst": args.n_inst, "seed": args.seed,
            "newton_iterations": int(iters), "accepted_steps": int(steps_acc),
            "failed_instances": len(bad),
            "batch_kernel": "lds" if batch.kernel == L.BATCH_KERNEL_LDS else "global",
            "launches": batch.n_launches,
        },
        "device_evals_per_s": n_mos_tot / (kernel_ms * 1e-3),
        "roofline": {
            "bound": "hbm",
            "achieved": achieved / 1e9,
            "peak": HBM_PEAK / 1e9,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK,
            "traffic": (measured("k_tran_pack_ring_mc_4096x10ns", "hbm_bytes_per_launch")
                        if (args.n_inst, args.t_stop, args.seed) == (4096, 10e-9, 2024)
                        and batch.kernel == L.BATCH_KERNEL_LDS else None),
            "kernel": "k_tran_pack" if batch.kernel == L.BATCH_KERNEL_LDS else "k_tran_batch",
            "kernel_ms": kernel_ms,
            "alg_bytes_per_launch": res.alg_bytes,
            "alg_flops_per_launch": res.alg_flops,
        },
    }
    # latency roofline: every instance's own device time (clock read at the
    # start and end of its run) against the launch.  With every instance
    # resident from the start, the launch could not end before its slowest
    # instance; per Newton iteration the instance waits on the levels of its
    # LU + forward and backward substitution schedules, one after another.
    busy = np.array([st_.busy_s for st_ in res.stats])
    if batch.kernel == L.BATCH_KERNEL_LDS and busy.max() > 0:
        its = np.array([st_.newton_iters for st_ in res.stats], dtype=np.float64)
        lev = np.array([systems[inst_sys[i]].info.lu_levels + systems[inst_sys[i]].info.bwd_levels
                        for i in range(args.n_inst)], dtype=np.float64)
        us_it = busy * 1e6 / np.maximum(its, 1)
        sel = {int(nst): stages == nst for nst in (int(stages.min()), int(stages.max()))}
        out["latency"] = {
            "critical_path_ms": float(busy.max() * 1e3),
            "kernel_ms": kernel_ms,
            "frac": float(busy.max() * 1e3 / kernel_ms),
            "mean_instance_ms": float(busy.mean() * 1e3),
            "us_per_newton_iter": {str(k): float(np.median(us_it[m])) for k, m in sel.items()},
            "levels_per_newton_iter": {str(k): float(np.median(lev[m])) for k, m in sel.items()},
            "us_per_level": {str(k): float(np.median(us_it[m] / lev[m])) for k, m in sel.items()},
        }
        log(f"latency: slowest instance {busy.max() * 1e3:.1f} ms of the {kernel_ms:.1f} ms launch; "
            f"us/iter {out['latency']['us_per_newton_iter']}")
    batch.close()

    if not args.no_plain and args.plain_sample > 0:
        # plain per-instance path over the full span, on the first instances
        idx = list(range(args.plain_sample))
        popts = dataclasses.replace(opts, batch_kernel=L.BATCH_KERNEL_GLOBAL)   # cs_tran's plain path
        t0 = time.perf_counter()
        for i in idx:
            s = systems[inst_sys[i]]
            sol = s.tran(popts, params[i], u0s[i])
            if sol.retcode != "Success":
                log(f"plain instance {i} failed: {sol.retcode}")
        dt = time.perf_counter() - t0
        plain = len(idx) / dt
        out["plain"] = {"value": plain, "unit": "instances/s",
                        "sample": f"{len(idx)} instance(s) (N={[int(stages[i]) for i in idx]}), "
                                  f"full 0-{args.t_stop * 1e9:g} ns each"}
        out["batched_vs_plain"] = value / plain
        log(f"plain: {plain:.4f} inst/s ({dt:.1f} s)")

    if not args.no_cpu:
        from oracle import oracle as O
        nproc, model = host_cpu()
        # the host cores this GPU's job may use (OMP_NUM_THREADS on a shared
        # box), else all of them
        thr = args.cpu_threads or int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or nproc
        k = min(args.cpu_sample or 4 * thr, args.n_inst)
        # size-stratified: every (n_inst/k)-th instance in stage-count order
        order = np.argsort(stages, kind="stable")
        pick = [int(order[int((j + 0.5) * args.n_inst / k)]) for j in range(k)]
        O.set_sparse(True)
        t0 = time.perf_counter()
        w, uf, st, rc = O.tran_batch([flats[i] for i in pick], [params[i] for i in pick],
                                     [u0s[i] for i in pick], opts, nthreads=thr)
        dt = time.perf_counter() - t0
        O.set_sparse(False)
        out["cpu_baseline"] = {"value": k / dt, "unit": "instances/s", "cores": thr, "kind": "port",
                               "nproc": nproc, "cpu_model": model,
                               "sample": f"{k} instances ({k // thr} per thread) of the same seeded batch, "
                                         f"size-stratified (every {args.n_inst / k:g}-th by stage count, "
                                         f"N {int(stages[pick].min())}-{int(stages[pick].max())}), full "
                                         f"0-{args.t_stop * 1e9:g} ns, OpenMP across instances, "
                                         f"sparse left-looking LU (oracle/sparse.c)"}
        log(f"cpu: {k / dt:.3f} inst/s ({dt:.1f} s, {thr} threads of {nproc}, {model}, rc {rc})")
    if args.adjoint_inst > 0:
        out["adjoint"] = adjoint_section(ch, L, ring_widths, args, eng)
    if args.bsim_inst > 0:
        out["device_eval"] = bsim_section(ch, args, eng)
    if args.grid_n > 0:
        out["power_grid"] = grid_section(ch, L, args, eng)
    eng.close()
    print(json.dumps(out), flush=True)


def adjoint_section(ch, L, ring_widths, args, eng):
    """Adjoint workload: n copies of a 51-stage ring, W ~ U[0.5, 4] um for all
    102 transistors, objective = supply energy over 0-5 ns, gradient w.r.t.
    every width, checkpoints every 64 accepted steps.  Timed: forward
    (recording) + reverse kernels, inputs uploaded inside the call."""
    n = args.adjoint_inst or 1024
    flats, params, u0s = ring_widths(n_inst=n, nstage=51, seed=args.seed)
    o = ch.TranOptions(t_start=0.0, t_stop=5e-9, reltol=1e-6, abstol=1e-9, newton_tol=1e-6,
                       newton_maxit=30, init=L.INIT_UIC)
    log(f"adjoint: {n} x 51-stage rings, 0-5 ns")
    t0 = time.perf_counter()
    try:
        res = ch.adjoint_batch(flats, params, u0s, o, vsrc=0, ckpt_every=64, max_steps=300_000,
                               engine=eng)
    except ch.CedarHIPError as e:
        log(f"adjoint unavailable: {e}")
        return {"error": str(e)}
    dt = time.perf_counter() - t0
    ok = sum(1 for r in res.retcodes if r == "Success")
    log(f"adjoint: {dt:.2f} s wall, kernels {res.kernel_ms:.1f} ms, {ok}/{n} ok, "
        f"mean steps {float(res.n_steps.mean()):.0f}")
    return {"value": n / (res.kernel_ms * 1e-3), "unit": "gradient instances/s",
            "kernel_ms": res.kernel_ms, "wall_s": dt, "n_inst": n, "ok": ok,
            "mean_steps": float(res.n_steps.mean()),
            "workload": "51-stage ring, W~U[0.5,4]um (102 widths), supply energy 0-5 ns, "
                        "dE/dW by discrete adjoint, checkpoint every 64 steps"}


def grid_section(ch, L, args, eng):
    """Power-grid workload on the supernodal path: n x n RC mesh (R ~ U[0.5,2]
    ohm, C ~ U[1,10] fF), inverters on random nodes driven by 1 ns square waves
    at random phases over the period (a phase in the second half written as the
    inverted pulse, so each pulse stays inside its period), VDD 1.0 V.  Times the symbolic analysis, the DC
    operating point, factorization and solve at the operating point (HIP
    events), and a transient over --grid-tstop (modified Newton by default:
    the step's first factorization serves its later iterations)."""
    from cedarhip.workloads import rc_mesh
    n = args.grid_n
    f = rc_mesh(n, n, args.grid_inv, seed=args.seed)
    t0 = time.perf_counter()
    s = eng.load(f, solver=L.SOLVER_SUPERNODAL)
    t_load = time.perf_counter() - t0
    bi = s.big_info
    log(f"grid: {n}x{n} mesh, {args.grid_inv} inverters, n {s.n}, {bi.n_super} fronts, "
        f"{bi.n_levels} levels, analysis+upload {t_load:.2f} s")
    p = f.params()
    t0 = time.perf_counter()
    dc = s.dcop(p)
    t_dc = time.perf_counter() - t0
    u = np.asarray(dc.u)
    A = s.jac_matrix(None, u, p, 1e12, 0.0)
    b = np.random.default_rng(args.seed).standard_normal(s.n)
    fms, sms = [], []
    for k in range(3):
        s.lu_refactor(A.data)
        s.lu_solve(b)
        fm, sm = s.lu_times()
        fms.append(fm)
        sms.append(sm)
    fm, sm = min(fms), min(sms)
    log(f"grid: dc {t_dc:.2f} s ({dc.retcode}), factor {fm:.3f} ms, solve {sm:.3f} ms")
    # per-launch HIP-event timing of the same factor + solve (plain stream
    # launches; per launch the minimum over three runs), summed by kernel
    runs = [s.profile() for _ in range(3)]
    prof = {}
    for q, (kind, lev, _) in enumerate(runs[0]):
        t = min(r[q][2] for r in runs)
        e = prof.setdefault(kind, {"launches": 0, "ms": 0.0})
        e["launches"] += 1
        e["ms"] += t
    for kind, e in sorted(prof.items(), key=lambda kv: -kv[1]["ms"]):
        log(f"grid: launches {kind:8s} {e['launches']:4d}  {e['ms']:8.3f} ms")
    o = ch.TranOptions(t_start=0.0, t_stop=args.grid_tstop, reltol=1e-6, abstol=1e-9,
                       jac_reuse=1 if args.grid_newton == "modified" else 0)
    t0 = time.perf_counter()
    sol = s.tran(o, p)
    wall = time.perf_counter() - t0
    st = sol.stats
    log(f"grid: transient 0-{args.grid_tstop * 1e9:g} ns {sol.retcode}: {st.steps} steps, "
        f"{st.newton_iters} Newton iterations, {wall:.2f} s")
    return {"value": args.grid_tstop * 1e9 / wall, "unit": "simulated ns/s",
            "n_unknowns": s.n, "fronts": bi.n_super, "levels": bi.n_levels, "max_front": bi.max_front,
            "factor_ms": fm, "solve_ms": sm, "factor_flops": bi.flops,
            "roofline": {"bound": "fp64 matrix", "achieved": bi.flops / (fm * 1e-3) / 1e12,
                         "peak": FP64_PEAK / 1e12, "unit": "TFLOP/s",
                         "frac": bi.flops / (fm * 1e-3) / FP64_PEAK, "kernel": "factorization (k_mf_*)",
                         "traffic": None},
            "factor_tflops": bi.flops / (fm * 1e-3) / 1e12, "fp64_peak_tflops": FP64_PEAK / 1e12,
            "factor_bytes_pool": 8 * bi.pool, "dcop_s": t_dc, "analysis_s": t_load,
            "launch_profile_ms": {k: round(e["ms"], 4) for k, e in prof.items()},
            "launch_counts": {k: e["launches"] for k, e in prof.items()},
            "tran_retcode": sol.retcode, "tran_steps": int(st.steps), "tran_newton_iters": int(st.newton_iters),
            "tran_wall_s": wall, "ms_per_newton_iter": wall * 1e3 / max(int(st.newton_iters), 1),
            "workload": f"{n}x{n} RC mesh + {args.grid_inv} square-law inverters (1 ns square-wave inputs at "
                        f"random phases over the period on a 10 ps grid), VDD 1.0 V, 0-{args.grid_tstop * 1e9:g} ns, "
                        "BDF2 reltol 1e-6, " + ("modified Newton" if o.jac_reuse else "full Newton")}


def bsim_section(ch, args, eng):
    """Device-eval microbenchmark: n BSIM-CMG 107 instances at the default
    card, L ~ U[20,100] nm, NFIN ~ U{1..8}, Vgs ~ U[-0.2,1] V, Vds ~ U[0,1] V,
    Vbs = 0; outputs I, Q (4) and the condensed 4x4 G, C per instance.  The
    value is evaluations/s of the kernel (inputs resident in HBM, HIP events
    around the launch); the wall rate including the PCIe copies is reported
    beside it."""
    if not ch.bsimcmg_available(eng):
        log("BSIM-CMG not in this build")
        return {"error": "library built without the generated BSIM-CMG model"}
    n = args.bsim_inst
    rng = np.random.default_rng(args.seed)
    Lg = rng.uniform(20e-9, 100e-9, n)
    nf = rng.integers(1, 9, n).astype(np.float64)
    v = np.zeros((n, 4))
    v[:, 0] = rng.uniform(0.0, 1.0, n)
    v[:, 1] = rng.uniform(-0.2, 1.0, n)
    log(f"bsim: {n} instances")
    r = ch.bsimcmg_eval(Lg, nf, v, engine=eng)            # warmup (module load, card upload)
    kms, walls = [], []
    for k in range(max(args.steps, 1)):
        t0 = time.perf_counter()
        r = ch.bsimcmg_eval(Lg, nf, v, engine=eng)
        walls.append(time.perf_counter() - t0)
        kms.append(r.kernel_ms)
        log(f"bsim step {k}: kernel {r.kernel_ms:.2f} ms, wall {walls[-1] * 1e3:.1f} ms")
    kernel_ms = float(np.mean(kms))
    evals = int(np.sum(r.iters + 1))                     # model evaluations incl. internal Newton
    fl = measured("k_bsimcmg_c1_1m", "fp64_flops_per_instance")
    out = {"value": n / (kernel_ms * 1e-3), "unit": "device evals/s", "n": n,
           "kernel": "k_bsimcmg", "kernel_ms": kernel_ms,
           "roofline": None if fl is None else {
               "bound": "fp64 valu", "achieved": fl * n / (kernel_ms * 1e-3) / 1e12, "peak": FP64_PEAK / 1e12,
               "unit": "TFLOP/s", "frac": fl * n / (kernel_ms * 1e-3) / FP64_PEAK,
               "traffic": measured("k_bsimcmg_c1_1m", "hbm_bytes_per_launch"),
               "flops_per_instance": fl},
           "wall_incl_pcie_evals_per_s": n / float(np.mean(walls)),
           "model_evals_per_instance": evals / n,
           "failed": int(np.sum(r.iters <= 0)),
           "workload": "BSIM-CMG 107 default card, L~U[20,100]nm, NFIN~U{1..8}, "
                       "Vgs~U[-0.2,1], Vds~U[0,1], Vbs=0, FP64, terminal I,Q,G(4x4),C(4x4)"}
    if not args.no_cpu:
        from oracle import oracle as O
        if O.va_lib() is not None:
            nproc, model = host_cpu()
            thr = args.cpu_threads or int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or nproc
            O.bsim_terminal_c(Lg[:1024], nf[:1024], v[:1024], nthreads=thr)     # warm the threads
            t0 = time.perf_counter()
            O.bsim_terminal_c(Lg, nf, v, nthreads=thr)
            dt = time.perf_counter() - t0
            out["cpu_baseline"] = {"value": n / dt, "unit": "device evals/s", "cores": thr,
                                   "kind": "port", "nproc": nproc, "cpu_model": model,
                                   "sample": f"all {n} instances of the same seeded set; the generated "
                                             "model compiled by g++ -O2 for the host, the bias-"
                                             "independent part once per instance, internal-node Newton "
                                             "and condensation in C++ (oracle/va_bsimcmg.cpp), OpenMP "
                                             "across instances"}
            log(f"bsim cpu: {n / dt:.0f} evals/s ({dt:.1f} s, {thr} threads)")
    return out


if __name__ == "__main__":
    main()
