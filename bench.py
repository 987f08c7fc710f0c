#!/usr/bin/env python3
"""Benchmark: Rayleigh-Benard timesteps/s at 256^2 x 129 Fourier-Chebyshev, FP64.

Workload (one MI355X): rotating Rayleigh-Benard convection in Coral's
primitive-variable form (coral_amd/inputs/coral.equations.rrbc_ra5e7_ek1e-4:
Ek = 1e-4, Ra = 5e7, Pr = 1), box 2pi x 2pi x 1, NX = NY = 256, NZ = 129
(padded grid 384 x 384 x 193), ARS_222, fixed dt = 2e-5, seeded temperature
perturbation on |k| <= 32 and the 8 lowest Galerkin modes, of amplitude 1e-30
so that the run stays within the advective CFL bound (see WORKLOADS).
A step is one full ARS_222 step (two implicit stages: transforms, products,
NL assembly, right-hand sides, banded solves).  State and operators are
resident in HBM before the timed region.

Prints one JSON line (see the bench contract in the repository notes):
metric/value (timesteps/s), roofline of the dominant kernel from HIP events on
the library's stream, and a CPU baseline from the oracle on the host cores.
"""
import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "RB timesteps/s at 256²×129 FP64; sim-time/s vs plain GPU at fixed Nu error"
PEAK_HBM_GBS = 8000.0
PEAK_FP64_TFLOPS = 78.6   # MI355X dense FP64 (matrix)

WORKLOADS = {
    # amplitude: the stated 1e-2 leaves the advective CFL bound of dt = 2e-5
    # within ~25 steps (linear growth ~1.14x per step at Ra = 5e7); 1e-30 keeps
    # every one of the 505 steps below it (CFL dt ~1e-4 at the end)
    "rrbc256": dict(eq="coral.equations.rrbc_ra5e7_ek1e-4", NX=256, NZ=129, dt=2e-5, amp=1e-30, kmax=32,
                    nmodes=8, seed=2, steps=500,
                    name="rotating RBC Ek=1e-4 Ra=5e7 Pr=1, 256x256x129 (384x384x193 padded), ARS_222, dt=2e-5"),
    "rbc64": dict(eq="coral.equations.rbc_ra1e5", NX=64, NZ=33, dt=1e-4, amp=1e-3, kmax=8, nmodes=8, seed=1,
                  steps=1000, name="RBC Ra=1e5 Pr=1, 64x64x33 (96x96x49 padded), ARS_222, dt=1e-4"),
    # the FP64 path at 512x512x257 (768x768x385 padded): rotating RBC, Ek=3e-5,
    # Ra=2e8, Pr=1, dt=5e-6
    "rrbc512": dict(eq="coral.equations.rrbc_ra2e8_ek3e-5", NX=512, NZ=257, dt=5e-6, amp=1e-30, kmax=64,
                    nmodes=8, seed=4, steps=20,
                    name="rotating RBC Ek=3e-5 Ra=2e8 Pr=1, 512x512x257 (768x768x385 padded), ARS_222, dt=5e-6"),
    # the case of Coral's own published timing: rotating RBC, Pr=1, Ra=2.81e5,
    # 1/Ek=707.1, 96x96x48 modes on a 2x2x1 box, 0.27 s per ARS_222 step on 20
    # Skylake cores (etc/benchmarks/02_RRBC_julien_JFM96/benchmark_02_RRBC_julien96.ipynb:78,
    # coral.parameters.in:2-4,14 there).  The case steps adaptively up to dt = 1e-3;
    # here dt is fixed at 1e-4, which keeps the seeded perturbation below the
    # advective CFL bound for all timed steps (the work of a step does not
    # depend on dt)
    "julien96": dict(eq="coral.equations.rrbc_ra2.81e5_iek707", NX=96, NZ=48, L=2.0, dt=1e-4, amp=1e-30, kmax=8,
                     nmodes=8, seed=3, steps=500, published_s_per_step=0.27,
                     name="rotating RBC Ek=1/707.1 Ra=2.81e5 Pr=1, 96x96x48 (144x144x72 padded), box 2x2x1, "
                          "ARS_222, dt=1e-4"),
}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def solve_bytes(N, nsys, real, blocks, u_entries, nfactored=None):
    """Algorithmic HBM bytes of one banded-solve launch.  Each of nfactored
    systems (all nsys of them unless symmetries let related wavenumbers share
    one factorization) is factored
    as nblk structural blocks of blk_n unknowns with band (bl, bu): per column
    bl multipliers, u_entries U entries (the mean length of the U records,
    each cut to the longest nonzero prefix its column has over all
    wavenumbers; at most bl+bu+1), 8 B per entry in real form, 16 B complex,
    and a 1 B pivot offset; per unknown the complex right-hand side read and
    the solution written.  (Row/column maps and rotation codes are shared by
    all systems and not counted.)"""
    nblk, blk_n, bl, bu = blocks
    e = 8 if real else 16
    nfac = nsys if nfactored is None else nfactored
    return int(nfac * nblk * blk_n * (e * bl + e * u_entries + 1) + nsys * N * (16 + 16))


def kernel_bytes(name, P):
    """Algorithmic bytes per launch of the main kernels (complex = 16 B, real = 8 B)."""
    N, nsys, NZ, NZAA, NYAA, nkx = P["N"], P["nsys"], P["NZ"], P["NZAA"], P["NYAA"], P["nkx"]
    nf, nq = P["nfull"], P["nquad"]
    S_sys = 16 * N * nsys
    table = {
        "solve": solve_bytes(N, nsys, P["real"], P["blocks"], P["u_entries"], P.get("nfactored")),
        # M (a x^n + b x_1) + K_hat terms: ARS_222 reads 2 (stage 1) and 4 (stage 2)
        # state vectors and writes one, 4 on average per launch
        "rhs": 4 * S_sys,
        "extract": S_sys + nf * 16 * NZ * nsys,              # state read, spectra written
        "zbwd": nf * 16 * (NZ + NZAA) * nsys,
        "ybwd": nf * 16 * NZAA * (nsys + NYAA * nkx),
        "xpass": 16 * NZAA * NYAA * nkx * (nf + nq),
        "yfwd": nq * 16 * NZAA * (nsys + NYAA * nkx),
        "zfwd": nq * 16 * (NZ + NZAA) * nsys,
        "nl_assemble": nq * 16 * NZ * nsys + S_sys,
    }
    return table.get(name)


def kernel_flops(name, P):
    """Floating-point operations per launch of the z transforms as executed on
    FP64 MFMA: each of the re/im columns of every (quadratic or full) variable
    and wavenumber is a product with the NZ x NZAA Chebyshev matrix, folded
    into even and odd halves (half of 2*NZ*NZAA)."""
    flops = {"zfwd": P["nquad"], "zbwd": P["nfull"]}
    if name not in flops:
        return None
    return flops[name] * 2 * P["nsys"] * P["NZ"] * P["NZAA"]


def cpu_baseline(wl, recipe, k0, z0, nsteps=1):
    """Oracle (numpy/scipy + OpenMP C) on the host cores: time `nsteps` steps after setup."""
    from oracle import coral_oracle as O
    L = wl.get("L", 2 * math.pi)
    geo = O.Geometry(wl["NX"], wl["NX"], wl["NZ"], L, L)
    ora = O.OracleSolver(recipe, geo, "ARS_222")
    ora.field, ora.zfield = [a.copy() for a in k0], [a.copy() for a in z0]
    t0 = time.perf_counter()
    ora.factorize(wl["dt"])
    t_setup = time.perf_counter() - t0
    t0 = time.perf_counter()
    for _ in range(nsteps):
        ora.step(wl["dt"])
    dt = time.perf_counter() - t0
    return nsteps / dt, t_setup, dt


def bench_ensemble(args):
    """Config 3: 48 independent Rayleigh-Benard runs drawn from a seed (NX = NY
    in {64, 96, 128}, NZ in {33, 49, 65}, Ra log-uniform in [1e5, 1e7], Pr in
    {0.7, 1, 7}, each with its own operators and dt), stepped as one ensemble
    (one HIP graph launch per step, tuned launch shapes and branches), against
    the same runs stepped one after another on their own (each with its own
    step graphs).  Every run's state after the ensemble steps is compared with
    its solo state."""
    import numpy as np
    from coral_amd import ensemble as E
    from coral_amd.ic import rbc_initial_state
    from coral_amd.solver import Solver
    nrun, seed = 48, 3
    steps = args.steps if args.steps is not None else 200
    specs = E.draw_runs(nrun, seed)
    t0 = time.perf_counter()
    runs = []
    for sp in specs:
        r = E.rbc_recipe(sp.Ra, sp.Pr)
        k0, z0 = rbc_initial_state(r, sp.NX, sp.NX, sp.NZ, 1e-4, 8, 6, sp.seed)
        g = Solver(r, sp.NX, sp.NX, sp.NZ, 2 * math.pi, 2 * math.pi)
        g.set_state(k0, z0)
        g.factorize_operators(sp.dt)
        runs.append((g, sp, k0, z0))
        if len(runs) % 8 == 0:
            log(f"ensemble: {len(runs)} runs created ({time.perf_counter() - t0:.1f} s)")
    # solo: each run alone, step graphs, one after another
    solo_ms, solo_state = [], []
    for g, sp, k0, z0 in runs:
        g.use_graphs(True)
        g.march_forward(sp.dt, 2)
        g.set_state(k0, z0)
        g.synchronize()
        t0 = time.perf_counter()
        g.march_forward(sp.dt, steps)
        g.synchronize()
        solo_ms.append(1e3 * (time.perf_counter() - t0) / steps)
        solo_state.append(g.get_state())
        g.use_graphs(False)
        g.set_state(k0, z0)
    solo_total = sum(solo_ms)
    log(f"solo runs one after another: {solo_total:.3f} ms per step of all runs")
    with E.Ensemble([g for g, _, _, _ in runs]) as ens:
        t0 = time.perf_counter()
        nb, tuned_ms = ens.tune(6)
        sched = f"lockstep, fronts over {-nb} branches" if nb <= 0 else f"{nb} branches"
        log(f"tuner: {sched}, {tuned_ms:.3f} ms per ensemble step, {time.perf_counter() - t0:.1f} s")
        ens.step(2)
        for g, _, k0, z0 in runs:
            g.set_state(k0, z0)
        ens.synchronize()
        t0 = time.perf_counter()
        ens.step(steps)
        ens.synchronize()
        elapsed = time.perf_counter() - t0
    worst, finite = 0.0, True
    for (g, _, _, _), (ks, zs) in zip(runs, solo_state):
        k, z = g.get_state()
        for a, b in zip(k + z, ks + zs):
            finite = finite and bool(np.isfinite(a).all())
            worst = max(worst, float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)))
    shapes = {}
    for g, sp, _, _ in runs:
        shapes.setdefault(f"{sp.NX}x{sp.NZ}", []).append(list(g.launch_shape()))
    value = steps / elapsed
    sim = sum(sp.dt for _, sp, _, _ in runs)
    out = {
        "metric": "ensemble steps/s (one step of every run), 48 uneven Rayleigh-Benard runs, FP64",
        "value": round(value, 3), "unit": "ensemble steps/s", "n_gpus": 1, "steps": steps,
        "ms_per_step": round(1e3 * elapsed / steps, 4), "higher_is_better": True, "dtype": "f64",
        "data": "synthetic (seeded perturbations)",
        "config": {"workload": f"{nrun} RBC runs drawn from seed {seed}: NX=NY in {{64,96,128}}, NZ in {{33,49,65}}, "
                               "Ra log-uniform [1e5,1e7], Pr in {0.7,1,7}, dt = 5e-5 (Ra Pr/1e5)^-1/2, ARS_222",
                   "runs": [[sp.NX, sp.NZ, round(sp.Ra, 1), sp.Pr, sp.dt] for _, sp, _, _ in runs],
                   "branches": nb, "schedule": sched, "launch_shapes": shapes},
        "run_steps_per_s": round(nrun * value, 1),
        "solo_sequential": {"ms_per_step_all_runs": round(solo_total, 4), "ensemble_steps_per_s": round(1e3 / solo_total, 3),
                            "per_run_ms": [round(x, 4) for x in solo_ms]},
        "speedup_vs_solo": round(value * solo_total / 1e3, 3),
        "sim_time_per_s": {"ensemble": round(value * sim, 6), "solo_sequential": round(1e3 / solo_total * sim, 6)},
        # the solo runs use the MFMA z transforms; a run the tuner moved to the
        # vector-GEMM ones (launch shape z_plain) matches its solo state to
        # rounding instead of bit for bit
        "parity_vs_solo": {"steps": steps, "worst_rel_l2": worst, "finite": finite,
                           "runs_on_vector_gemm_z": sum(1 for g, _, _, _ in runs if g.launch_shape()[1])},
    }
    print(json.dumps(out), flush=True)


def bench_mixed(args):
    """Config 4: the rotating 512^2 x 257 workload (Ek = 3e-5, Ra = 2e8, Pr = 1,
    dt = 5e-6, 300 steps) in FP64 and in mixed precision (FP32 transforms and
    products, FP64 solves, one FP64 refinement sweep per step) from the same
    seeded state: sim-time/s of both, and the mixed run's errors against the
    FP64 run in kinetic energy (the volume average of uu + vv + ww, Coral's
    KE_display), the Nusselt number (compute_nusselt.py's wall estimator on
    the mean temperature) and the horizontal spectrum of the velocity state."""
    import numpy as np
    from coral_amd import diagnostics as D
    from coral_amd.equations import read_equations
    from coral_amd.ic import interleaved_positions, rbc_initial_state
    from coral_amd.solver import Solver
    wl = WORKLOADS["rrbc512"]
    steps = args.steps if args.steps is not None else 300
    # amplitude: the perturbation grows about 4x per 25 steps at this Ra and dt;
    # from 1e-8 the CFL time step falls below dt near step 250, from 1e-11 the
    # 300 steps stay inside it (the final CFL time step is reported)
    amp = args.amp if args.amp is not None else 1e-11
    recipe = read_equations(os.path.join(ROOT, "coral_amd", "inputs", wl["eq"]))
    NX, NZ, dt = wl["NX"], wl["NZ"], wl["dt"]
    k0, z0 = rbc_initial_state(recipe, NX, NX, NZ, amp, wl["kmax"], wl["nmodes"], wl["seed"])
    s = recipe.kxky_systems[0]
    sizes = [NZ - bc // 10 for bc in s.bc_codes]
    vel = np.concatenate([interleaved_positions(len(sizes), sizes, s.var_names.index(v)) for v in ("u", "v", "w")])
    tsys = [i for i, z in enumerate(recipe.zero_systems) if "tMean" in z.var_names][0]
    tvar = recipe.zero_systems[tsys].var_names.index("tMean")
    res = {}
    with Solver(recipe, NX, NX, NZ, 2 * math.pi, 2 * math.pi) as g:
        diag = D.Diagnostics(g)
        for mode, refine in (("fp64", 0), ("mixed", 0), ("mixed_refined", 1)):
            g.set_precision("mixed" if mode != "fp64" else "fp64", refine)
            g.use_graphs(True)
            g.set_state(k0, z0)
            g.factorize_operators(dt)
            g.march_forward(dt, 2)
            g.set_state(k0, z0)
            g.synchronize()
            t0 = time.perf_counter()
            g.march_forward(dt, steps)
            g.synchronize()
            el = time.perf_counter() - t0
            _, ke = diag.sample()
            prof = g.variable_physical("zero", tsys, tvar)
            nu = D.nusselt_wall_differences(prof, g.gap)
            k, _ = g.get_state()
            spec = D.horizontal_spectrum(k[0], vel, NX, NX, 2 * math.pi, 2 * math.pi)
            res[mode] = dict(elapsed=el, ke=ke, nu=nu, spec=spec, cfl=g.cfl_dt(), finite=bool(np.isfinite(k[0]).all()))
            log(f"{mode}: {steps} steps in {el:.3f} s, KE {ke:.6e}, Nu (top, bottom) {nu}, CFL dt {res[mode]['cfl']:.3e}")
            g.use_graphs(False)
            # per-kernel figures of 10 eager steps
            g.timers_enable(True)
            g.march_forward(dt, 10)
            g.synchronize()
            res[mode]["kernels"] = {n: round(ms / 10, 3) for n, (ms, c) in g.timers().items()}
            g.timers_enable(False)
            log(f"{mode} kernels (ms per step): {res[mode]['kernels']}")
    a, b, ar = res["mixed"], res["fp64"], res["mixed_refined"]

    def errs(x):
        return {"kinetic_energy_rel": abs(x["ke"] / b["ke"] - 1),
                "nusselt_rel": max(abs(p / q - 1) for p, q in zip(x["nu"], b["nu"])),
                "horizontal_spectrum_rel_l2": float(np.linalg.norm(x["spec"] - b["spec"]) / np.linalg.norm(b["spec"]))}
    out = {
        "metric": "sim-time/s, mixed precision vs plain FP64 GPU, 512²×257 rotating RBC",
        "value": round(steps * dt / a["elapsed"], 8), "unit": "simulated time units/s", "n_gpus": 1, "steps": steps,
        "ms_per_step": round(1e3 * a["elapsed"] / steps, 4), "higher_is_better": True, "dtype": "f32 transforms, f64 solves",
        "data": "synthetic (seeded perturbation)",
        "config": {"workload": wl["name"] + f", {steps} steps", "ic_amplitude": amp, "refine": 0},
        "fp64": {"sim_time_per_s": round(steps * dt / b["elapsed"], 8), "ms_per_step": round(1e3 * b["elapsed"] / steps, 4),
                 "kernels_ms_per_step": b["kernels"]},
        "speedup_vs_fp64": round(b["elapsed"] / a["elapsed"], 4),
        "errors_vs_fp64": errs(a),
        "kernels_ms_per_step": a["kernels"],
        "mixed_refined": {"sim_time_per_s": round(steps * dt / ar["elapsed"], 8),
                          "ms_per_step": round(1e3 * ar["elapsed"] / steps, 4),
                          "speedup_vs_fp64": round(b["elapsed"] / ar["elapsed"], 4), "errors_vs_fp64": errs(ar)},
        "values": {"ke_fp64": b["ke"], "ke_mixed": a["ke"], "nu_fp64": b["nu"], "nu_mixed": a["nu"],
                   "cfl_dt_fp64": b["cfl"], "finite": a["finite"] and b["finite"] and ar["finite"]},
    }
    print(json.dumps(out), flush=True)


CLOSURE_WORKLOADS = {
    # learned closure, evaluated at 128^2 x 65 (the coarse grid of the
    # closure's target configuration) against a 256^2 x 129 fine run
    "closure128": dict(fine=(256, 129), coarse=(128, 65), spin=(128, 65, 12000, 3000), snapshots=42, every=25,
                       epochs=12, t_eval=0.02),
    # the same at half the size in every direction
    "closure64": dict(fine=(128, 65), coarse=(64, 33), spin=(128, 65, 12000, 0), snapshots=150, every=25,
                      epochs=20, t_eval=0.05),
}


def bench_closure(args, name):
    """Config 5 at reduced scale: Rayleigh-Benard convection at Ra = 1e6, Pr = 1
    (2pi x 2pi x 1 box, noisy start, adaptive dt: dt_max 1e-3, CFL 0.2).  A fine
    run spun up to the statistically steady state (on a coarser grid first
    when the workload says so, then embedded); snapshots of the fine run are
    box-filtered (top-hat over one coarse cell) onto the coarse grid and give
    the training pairs (the filtered full variables on each point's 3 x 3 x 3
    neighbourhood -> the subgrid part of every quadratic variable); the
    network (--closure-width, --closure-hidden; 4 layers, modes |k| <= 4) is trained on the
    first 5/6 of the snapshots and scored on the rest (relative L2 error; 1 =
    no closure).  Then, from the filtered final fine state, the fine run, the
    plain coarse run and the coarse run with the closure each advance t_eval
    time units: Nusselt numbers (mean of the wall estimator every 50 steps) and
    simulated time per second of each.  The metric is the closure run's
    sim-time/s; its Nu error against the fine run beside the plain coarse
    run's."""
    import numpy as np
    from coral_amd import closure as CL
    from coral_amd import ic
    from coral_amd.diagnostics import gauss_chebyshev_grid
    from coral_amd.ensemble import rbc_recipe
    from coral_amd.solver import Solver
    from coral_amd.timekeeping import Timings
    wl = CLOSURE_WORKLOADS[name]
    Ra, L = 1e6, 2 * math.pi
    r = rbc_recipe(Ra, 1.0)
    (NXf, NZf), (NXc, NZc) = wl["fine"], wl["coarse"]
    NXs, NZs, nspin, nspin_fine = wl["spin"]
    tsys = [i for i, z in enumerate(r.zero_systems) if "tMean" in z.var_names][0]
    tvar = r.zero_systems[tsys].var_names.index("tMean")

    def nusselt(g):
        p = g.variable_physical("zero", tsys, tvar)
        dz = 0.5 * (1 - math.cos(math.pi / (2 * p.size)))
        return 0.5 * (p[0] - p[-1]) / dz

    def advance(g, tk, n):
        for _ in range(n):
            tk.check_for_update()
            if tk.refactorization_is_due:
                g.factorize_operators(tk.dt_current)
                tk.refactorization_is_due = False
            g.march_forward(tk.dt_current, 1)
            tk.apply_cfl(g.cfl_dt())
            tk.increment()

    t_all = time.perf_counter()
    tk = Timings(1e-3, 0.3, 0.2)
    gs = Solver(r, NXs, NXs, NZs, L, L)
    gs.use_graphs(True)
    gs.set_kx0_projection(True)
    k0, z0 = ic.noisy_initial_state(r, NXs, NXs, NZs, L, L, 1e-2, 1e-2, 5)
    gs.set_state(k0, z0)
    for i in range(nspin // 1000):
        advance(gs, tk, 1000)
        log(f"closure: spin-up {1000 * (i + 1)} steps at {NXs}x{NZs}, t = {tk.absolute_time:.4f}, Nu = {nusselt(gs):.3f}")
    if (NXs, NZs) != (NXf, NZf):
        k, z = gs.get_state()
        gs.close()
        gf = Solver(r, NXf, NXf, NZf, L, L)
        kf, zf = CL.BoxFilter(r, (NXf, NXf, NZf), (NXs, NXs, NZs), kind="sharp").embed(k, z)
        gf.set_state(kf, zf)
        tk.refactorization_is_due = True
    else:
        gf = gs
    gf.use_graphs(True)
    gf.set_kx0_projection(True)
    for i in range(nspin_fine // 500):
        advance(gf, tk, 500)
        log(f"closure: spin-up {500 * (i + 1)} steps at {NXf}x{NZf}, t = {tk.absolute_time:.4f}, Nu = {nusselt(gf):.3f}")
    gc = Solver(r, NXc, NXc, NZc, L, L)
    box = CL.BoxFilter(r, (NXf, NXf, NZf), (NXc, NXc, NZc))
    zg = gauss_chebyshev_grid(3 * NZc // 2, 0.5, 1.0)
    X, T = [], []
    t0 = time.perf_counter()
    for i in range(wl["snapshots"]):
        advance(gf, tk, wl["every"])
        xi, ti = CL.subgrid_sample(gf, gc, box, zg)
        X.append(xi)
        T.append(ti)
        if (i + 1) % 16 == 0:
            log(f"closure: {i + 1} snapshots, t = {tk.absolute_time:.4f} ({time.perf_counter() - t0:.0f} s)")
    N2 = (3 * NXc // 2) ** 2
    nval = max(1, len(X) // 6)
    # per-snapshot arrays, never concatenated (a 128^2 x 65 snapshot is 1.6 GB of rows)
    Xtr, Ttr, Xva = X[:-nval], T[:-nval], X[-nval:]
    Tva = np.concatenate(T[-nval:])
    basis = CL.fourier_basis(3 * NXc // 2, 3 * NXc // 2, 4)
    t0 = time.perf_counter()
    model, hist = CL.train(Xtr, Ttr, N2, basis, 4, width=args.closure_width, hidden=args.closure_hidden,
                           epochs=wl["epochs"], planes_per_batch=16, lr=2e-3, log=log)
    t_train = time.perf_counter() - t0
    pred = CL.predict(model, Xva, N2, basis)
    del X, T, Xtr, Ttr, Xva
    err = np.linalg.norm(pred - Tva, axis=0) / np.linalg.norm(Tva, axis=0)
    err_all = float(np.linalg.norm(pred - Tva) / np.linalg.norm(Tva))
    log(f"closure: trained in {t_train:.1f} s; held-out relative L2 error {err_all:.3f} per variable {np.round(err, 3)}")
    kf, zf = gf.get_state()
    kc, zc = box.state(kf, zf)
    res = {}
    for run, g, use in (("fine", gf, None), ("coarse", gc, False), ("coarse_closure", gc, True)):
        if run != "fine":
            g.set_closure(model if use else None)
            g.set_kx0_projection(True)
            g.use_graphs(True)
            g.set_state(kc, zc)
        tke = Timings(1e-3, 0.3, 0.2)
        tke.absolute_time = 0.0
        nus, n = [], 0
        g.synchronize()
        t0 = time.perf_counter()
        while tke.absolute_time < wl["t_eval"]:
            advance(g, tke, 50)
            n += 50
            nus.append(nusselt(g))
            if not np.isfinite(nus[-1]):
                break
        el = time.perf_counter() - t0
        res[run] = dict(nu=float(np.mean(nus)), nu_std=float(np.std(nus)), steps=n, sim_per_s=tke.absolute_time / el,
                        ms_per_step=1e3 * el / n, finite=bool(np.all(np.isfinite(nus))))
        log(f"closure: {run}: Nu {res[run]['nu']:.4f} +- {res[run]['nu_std']:.4f} over {n} steps, "
            f"{res[run]['sim_per_s']:.5f} sim-time/s, {res[run]['ms_per_step']:.3f} ms/step")
    nu_f = res["fine"]["nu"]
    c = res["coarse_closure"]
    out = {
        "metric": "sim-time/s of the coarse run with the learned closure, vs the fine GPU run, at its Nu error",
        "value": round(c["sim_per_s"], 6), "unit": "simulated time units/s", "n_gpus": 1, "steps": c["steps"],
        "ms_per_step": round(c["ms_per_step"], 4), "higher_is_better": True,
        "dtype": "f64 solver, bf16 network (f32 accumulate)", "data": "synthetic (noisy start, self-generated training set)",
        "config": {"workload": f"RBC Ra=1e6 Pr=1, fine {NXf}^2x{NZf} -> coarse {NXc}^2x{NZc}, top-hat box filter, "
                               f"{wl['snapshots']} snapshots every {wl['every']} steps, {wl['epochs']} epochs, "
                               f"evaluation over {wl['t_eval']} time units",
                   "network": {"width": args.closure_width, "hidden": args.closure_hidden, "layers": 4, "modes": 4,
                               "params": int(model.layout.size)}},
        "vs_fine": round(c["sim_per_s"] / res["fine"]["sim_per_s"], 4),
        "nu_rel_error": {"coarse_closure": abs(c["nu"] / nu_f - 1), "coarse": abs(res["coarse"]["nu"] / nu_f - 1)},
        "a_priori_rel_l2": {"overall": err_all, "per_quadratic_variable": [round(float(e), 4) for e in err]},
        "runs": res, "training_s": round(t_train, 1), "wall_s": round(time.perf_counter() - t_all, 1),
    }
    print(json.dumps(out), flush=True)


def bench_closure_step(args):
    """The closure's inference cost inside the coarse step at 128^2 x 65 (the
    coarse grid of the closure configuration): RBC Ra = 1e6, the network with
    random weights (its cost does not depend on them), width and hidden from
    --closure-width / --closure-hidden (4 layers, modes |k| <= 4), 20 eager
    steps with per-kernel events after 3 warmup steps, against the same
    steps without the closure.  Reports ms per step with and without it and
    the closure's share by kernel group."""
    import numpy as np
    from coral_amd import closure as CL
    from coral_amd import ic
    from coral_amd.ensemble import rbc_recipe
    from coral_amd.solver import Solver
    NX, NZ, M = 128, 65, 4
    W, Hd = args.closure_width, args.closure_hidden
    steps = args.steps if args.steps is not None else 20
    r = rbc_recipe(1e6, 1.0)
    L = 2 * math.pi
    NXAA = 3 * NX // 2
    basis = CL.fourier_basis(NXAA, NXAA, M)
    cin = CL.input_width(len(r.full_vars))
    lay = CL.Layout(cin=cin, cout=len(r.quad_vars), width=W, hidden=Hd, layers=4, nb=basis.shape[1])
    model = CL.Model(lay, M, CL.init_params(lay, 1), np.zeros(cin), np.ones(cin), np.zeros(lay.cout),
                     np.full(lay.cout, 1e-3))
    res = {}
    with Solver(r, NX, NX, NZ, L, L) as g:
        k0, z0 = ic.noisy_initial_state(r, NX, NX, NZ, L, L, 1e-3, 1e-3, 5)
        g.factorize_operators(1e-5)
        for name, use in (("plain", False), ("closure", True)):
            g.set_state(k0, z0)
            g.set_closure(model if use else None)
            g.march_forward(1e-5, 3)
            g.synchronize()
            g.timers_enable(True)
            t0 = time.perf_counter()
            g.march_forward(1e-5, steps)
            g.synchronize()
            el = time.perf_counter() - t0
            res[name] = {"ms_per_step": round(1e3 * el / steps, 4),
                         "kernels_ms_per_step": {k: round(v[0] / steps, 4) for k, v in g.timers().items()}}
            g.timers_enable(False)
            log(f"{name}: {res[name]['ms_per_step']:.3f} ms/step, {res[name]['kernels_ms_per_step']}")
    out = {"metric": "coarse-step time with the learned closure, RBC 128^2x65", "value": res["closure"]["ms_per_step"],
           "unit": "ms/step", "n_gpus": 1, "steps": steps, "higher_is_better": False,
           "dtype": "f64 solver, bf16 network (f32 accumulate)", "data": "synthetic (random weights)",
           "config": {"workload": "RBC Ra=1e6 Pr=1, 128x128x65 (192x192x97 padded), ARS_222, eager with events",
                      "network": {"width": W, "hidden": Hd, "layers": 4, "modes": M, "params": int(lay.size)}},
           "plain_ms_per_step": res["plain"]["ms_per_step"], "runs": res}
    print(json.dumps(out), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=None)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="rrbc256",
                    choices=sorted(WORKLOADS) + ["ensemble48", "mixed512", "closure_step"] + sorted(CLOSURE_WORKLOADS),
                    help="ensemble48: 48 uneven runs as one ensemble against solo runs; mixed512: mixed precision "
                         "against FP64 at 512^2 x 257 (sim-time/s and KE, Nu, spectrum errors); closure128 / "
                         "closure64: a learned closure trained on a filtered fine run, coarse sim-time/s and Nu "
                         "error against the fine and the plain coarse runs")
    ap.add_argument("--closure-width", type=int, default=32, help="closure_step / closure*: network width")
    ap.add_argument("--closure-hidden", type=int, default=128, help="closure_step / closure*: MLP hidden width")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--eager-only", action="store_true",
                    help="skip the second timed pass of the same steps replayed as HIP graphs")
    ap.add_argument("--graphs", action="store_true",
                    help="time the steps replayed as HIP graphs (timers off); the per-kernel figures then come "
                         "from a separate eager pass of min(steps, 50) steps")
    ap.add_argument("--cpu-steps", type=int, default=1)
    ap.add_argument("--amp", type=float, default=None,
                    help="amplitude of the seeded temperature perturbation (default: the workload's)")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MIB",
                    help="only run a plain device-to-device copy of MIB MiB (5 times); its FETCH_SIZE/WRITE_SIZE "
                         "counters calibrate the per-kernel HBM traffic figures")
    args = ap.parse_args()
    if args.calibrate_copy:
        import torch
        n = args.calibrate_copy * (1 << 20) // 8
        src = torch.arange(n, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        log(f"copied {args.calibrate_copy} MiB 5 times")
        return
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build runs the whole domain on one GPU; multi-GPU runs are not part of it "
              "(the systems would shard by kx slabs, each transform with one all-to-all).", file=sys.stderr)
        sys.exit(2)
    if args.workload == "ensemble48":
        return bench_ensemble(args)
    if args.workload == "mixed512":
        return bench_mixed(args)
    if args.workload in CLOSURE_WORKLOADS:
        return bench_closure(args, args.workload)
    if args.workload == "closure_step":
        return bench_closure_step(args)
    wl = WORKLOADS[args.workload]
    steps = args.steps if args.steps is not None else wl["steps"]

    from coral_amd.equations import read_equations
    from coral_amd.ic import rbc_initial_state
    from coral_amd.solver import Solver
    import numpy as np

    recipe = read_equations(os.path.join(ROOT, "coral_amd", "inputs", wl["eq"]))
    NX, NZ = wl["NX"], wl["NZ"]
    amp = args.amp if args.amp is not None else wl["amp"]
    k0, z0 = rbc_initial_state(recipe, NX, NX, NZ, amp, wl["kmax"], wl["nmodes"], wl["seed"])
    L = wl.get("L", 2 * math.pi)
    g = Solver(recipe, NX, NX, NZ, L, L, scheme="ARS_222")
    total, kl, ku, nsys = g.system_info(0)
    g.set_state(k0, z0)
    t0 = time.perf_counter()
    g.factorize_operators(wl["dt"])
    log(f"setup: LU factorization of {nsys} systems (N={total}, kl={kl}, ku={ku}) in {time.perf_counter() - t0:.3f} s")
    g.march_forward(wl["dt"], args.warmup)
    g.synchronize()

    if args.graphs:
        # steps as HIP graph replays, timed without per-kernel events; then an
        # eager pass with events for the per-kernel figures
        g.use_graphs(True)
        g.march_forward(wl["dt"], 2)   # capture
        g.synchronize()
        t0 = time.perf_counter()
        g.march_forward(wl["dt"], steps)
        g.synchronize()
        elapsed = time.perf_counter() - t0
        g.use_graphs(False)
        ksteps = min(steps, 50)
        g.timers_enable(True)
        g.march_forward(wl["dt"], ksteps)
        g.synchronize()
        timers = g.timers()
        g.timers_enable(False)
    else:
        ksteps = steps
        g.timers_enable(True)
        g.synchronize()
        t0 = time.perf_counter()
        g.march_forward(wl["dt"], steps)
        g.synchronize()
        elapsed = time.perf_counter() - t0
        timers = g.timers()
        g.timers_enable(False)
    cfl_final = g.cfl_dt()
    kfin, _ = g.get_state()
    finite = bool(np.isfinite(kfin[0]).all())
    norm = float(np.linalg.norm(kfin[0]))
    log(f"{steps} steps in {elapsed:.3f} s, state finite={finite}, |state|={norm:.6e}, CFL dt of the last stage "
        f"{cfl_final:.3e} (dt {wl['dt']:.1e})")
    graphs_line = None
    if not args.graphs and not args.eager_only:
        # the same steps from the same state, replayed as HIP graphs (no
        # per-kernel events); reported beside the eager figure
        g.use_graphs(True)
        g.set_state(k0, z0)
        g.march_forward(wl["dt"], 2)   # capture
        g.set_state(k0, z0)
        t0 = time.perf_counter()
        g.march_forward(wl["dt"], steps)
        g.synchronize()
        gel = time.perf_counter() - t0
        kg, _ = g.get_state()
        g.use_graphs(False)
        graphs_line = {"value": round(steps / gel, 4), "ms_per_step": round(1e3 * gel / steps, 4), "steps": steps,
                       "state_finite": bool(np.isfinite(kg[0]).all())}
        log(f"{steps} steps as HIP graph replays in {gel:.3f} s")

    value_check = None
    if args.workload == "rrbc256" and not args.graphs:
        # the step's work does not depend on the values: the same 20 eager
        # steps from the stated amplitude 1e-2 (finite through step ~39) and
        # from the headline's amplitude
        vc = {}
        for a_ in (1e-2, amp):
            ka, za = rbc_initial_state(recipe, NX, NX, NZ, a_, wl["kmax"], wl["nmodes"], wl["seed"])
            g.set_state(ka, za)
            g.synchronize()
            t0 = time.perf_counter()
            g.march_forward(wl["dt"], 20)
            g.synchronize()
            kc, _ = g.get_state()
            vc[a_] = (1e3 * (time.perf_counter() - t0) / 20, bool(np.isfinite(kc[0]).all()))
        value_check = {"steps": 20, "launch": "eager, no events",
                       "amp_1e-2": {"ms_per_step": round(vc[1e-2][0], 4), "state_finite": vc[1e-2][1]},
                       f"amp_{amp:g}": {"ms_per_step": round(vc[amp][0], 4), "state_finite": vc[amp][1]}}
        log(f"value check: 20 steps at amplitude 1e-2 {vc[1e-2][0]:.3f} ms/step, at {amp:g} {vc[amp][0]:.3f} ms/step")

    P = dict(N=total, kl=kl, ku=ku, nsys=nsys, real=g.factor_is_real(0), blocks=g.factor_blocks(0),
             u_entries=g.u_entries_per_column(0), nfactored=g.factored_systems(0)[0], NZ=NZ,
             NZAA=3 * NZ // 2, NYAA=3 * NX // 2, nkx=NX // 2,
             nfull=len(recipe.full_vars), nquad=len(recipe.quad_vars))
    per_kernel = {}
    for name, (ms, cnt) in timers.items():
        per_kernel[name] = {"ms_per_launch": ms / cnt, "launches_per_step": cnt / ksteps,
                            "ms_per_step": ms / ksteps}
        b = kernel_bytes(name, P)
        if b is not None:
            per_kernel[name]["GBps"] = b / (ms / cnt * 1e-3) / 1e9
    for name, v in sorted(per_kernel.items(), key=lambda kv: -kv[1]["ms_per_step"]):
        log(f"  {name:14s} {v['ms_per_step']:9.3f} ms/step  {v['ms_per_launch']:8.3f} ms/launch"
            + (f"  {v['GBps']:8.1f} GB/s" if "GBps" in v else ""))
    # dominant kernel with an algorithmic byte count
    dom = max((n for n in per_kernel if kernel_bytes(n, P) is not None), key=lambda n: per_kernel[n]["ms_per_step"])
    dom_bytes = kernel_bytes(dom, P)
    achieved = dom_bytes / (per_kernel[dom]["ms_per_launch"] * 1e-3) / 1e9
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "traffic.json")
    if os.path.exists(tpath):
        tr = json.load(open(tpath)).get(args.workload, {}).get(dom)
        if tr is not None:
            traffic = tr.get("bytes_per_launch")
    roofline = {"bound": "hbm", "kernel": dom, "achieved": round(achieved, 2), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                "frac": round(achieved / PEAK_HBM_GBS, 4), "traffic": traffic, "algorithmic_bytes": dom_bytes}
    # per-kernel figures: algorithmic HBM GB/s of every main kernel, FP64 MFMA
    # rate and utilisation of the z transforms, banded-solve time per wavenumber
    kernels = {}
    for name, v in per_kernel.items():
        b, f = kernel_bytes(name, P), kernel_flops(name, P)
        if b is None:
            continue
        k = {"ms_per_launch": round(v["ms_per_launch"], 4), "GBps": round(v["GBps"], 1),
             "hbm_frac": round(v["GBps"] / PEAK_HBM_GBS, 4)}
        if f is not None:
            tf = f / (v["ms_per_launch"] * 1e-3) / 1e12
            k.update({"TFLOPs": round(tf, 2), "mfma_fp64_frac": round(tf / PEAK_FP64_TFLOPS, 4)})
        if name == "solve":
            k["ns_per_wavenumber"] = round(v["ms_per_launch"] * 1e6 / nsys, 2)
        kernels[name] = k

    cpu = None
    if not args.no_cpu_baseline:
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        try:
            v, t_setup, t_run = cpu_baseline(wl, recipe, k0, z0, args.cpu_steps)
            cpu = {"value": round(v, 5), "unit": "timesteps/s", "cores": threads, "kind": "port",
                   "sample": f"{args.cpu_steps} ARS_222 step(s) of the same workload by the oracle "
                             f"(numpy/scipy.fft with {threads} workers + OpenMP C banded LU) after setup; "
                             f"setup {t_setup:.1f} s excluded, timed {t_run:.1f} s"}
        except MemoryError as e:  # pragma: no cover
            cpu = {"value": None, "unit": "timesteps/s", "cores": threads, "kind": "port",
                   "sample": f"failed: {e}"}

    value = steps / elapsed
    out = {
        "metric": METRIC,
        "value": round(value, 4),
        "unit": "timesteps/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * elapsed / steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded perturbation, no checkpoint)",
        "launch": "hip graphs" if args.graphs else "eager, per-kernel events",
        "config": {"workload": wl["name"], "grid": [NX, NX, NZ], "systems": nsys, "unknowns_per_system": total,
                   "band": [kl, ku], "factors": "real form" if P["real"] else "complex",
                   "factored_blocks": {"per_system": P["blocks"][0], "unknowns": P["blocks"][1],
                                       "band": [P["blocks"][2], P["blocks"][3]],
                                       "u_entries_per_column": round(P["u_entries"], 3)},
                   "ic_amplitude": amp, "state_finite": finite, "cfl_dt_last_stage": cfl_final},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "kernels_ms_per_step": {k: round(v["ms_per_step"], 4) for k, v in per_kernel.items()},
        "kernels": kernels,
        "hip_graphs": graphs_line,
        "value_independence": value_check,
    }
    if "published_s_per_step" in wl:
        # Coral's own timing of this case (other hardware: 20 Skylake cores, MPI)
        pub = 1.0 / wl["published_s_per_step"]
        out["published_cpu_reference"] = {"s_per_step": wl["published_s_per_step"], "timesteps_per_s": round(pub, 3),
                                          "cores": 20, "hardware": "Intel Skylake, MPI",
                                          "gpu_over_published": round(value / pub, 1)}
        if graphs_line:
            out["published_cpu_reference"]["gpu_graphs_over_published"] = round(graphs_line["value"] / pub, 1)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
