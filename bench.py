"""Benchmark: Stokes solves/s to relative residual 1e-6 on one MI355X.

One step = one complete Stokes solve of the 1,013,958-velocity-dof shell
(level-4 icosahedral surface x 16 layers, 245,760 P2 tets, 3-level MG):
element assembly with rotation and BC elimination, element-local Galerkin
coarse operators, coarse Cholesky factorisation, Patera pressure iteration
with the MGPCG velocity solves, until
    rel_res = max(|r_P| / |r_P^cold|, |r_U| / |f_U|) <= 1e-6
(RMS norms; r_P^cold is the pressure residual of the velocity solve at P=0,
the same denominator for every form).  Inputs are seeded synthetic fields
(temperature with spherical-harmonic perturbation, viscosity contrast 1e4,
6 Voronoi plates at the surface, free slip at the CMB).

Forms:
  learned (default): the headline metric.  Input is a held-out time step k
    of the seeded c1 convection trajectory (vertex temperatures and times of
    steps k-3..k, shipped in m3tet_sph_amd/data).  Untimed: FP64 solves of
    steps k-3..k-1 to the same rel.res as the timed solves give the
    converged states that a time loop holds when it reaches step k; a cold
    FP64 solve of step k gives |r_P^cold|.  Timed,
    each as K solves after W warm-ups:
      plain FP64 MGPCG from a cold start (the reference solver as configured
        for a single solve: P = 0, U from the BCs);
      FP64 and mixed from the previous step (the reference's time loop warm
        start, flow3d_patera_mg_sph_p.m:204-231);
      FP64 and mixed from the quadratic extrapolation in time of the last
        three converged states (no network);
      FP64 + learned, and mixed precision + learned warm start: the
        extrapolation plus the network's correction, computed from
        (T, ln eta, the extrapolated state, T minus its extrapolation),
        followed by the solve;
    (the extrapolated and learned starts are formed on the GPU and handed to
    the solver there, m3_flow3d_patera_sph_dstart; the previous-step start
    comes from host memory, as the reference passes VAR to the solver)
    all stopping at the same fixed residual.  ``value`` is the mixed+learned
    rate; the others are reported beside it.
  fp64 / mixed: cold solves of the seed-0 temperature field.

Prints one JSON line.  Usage:
  python bench.py [--gpus 1] [--steps K] [--warmup W] [--config c1]
                  [--form learned|fp64|mixed] [--no-cpu]

``--path diffusion`` times the thermal diffusion step instead (not the
headline metric): diffusion3d_p on the linear tetrahedra of --config
(--grid vertex: the P1 vertex tetrahedra; p2split: every P2 element split
into 8), element matrices + lumped mass + backward-Euler system with the
CMB / surface temperatures fixed + Jacobi PCG to 1e-8, with the diffusivity
set so that kappa dt / h_min^2 = 1; its cpu_baseline is the same step in the
oracle.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

HBM_PEAK_GBS = 8000.0

# HBM bytes per launch of the dominant kernel, measured with two rocprofv3
# counter passes (FETCH_SIZE x 2.0000 + WRITE_SIZE x 1.0000, factors from the
# 1 GiB copy kernel of m3_copy_rate profiled in the same runs); recorded in
# profiles/c1_sweep_hbm_traffic.md.  Keyed by (config, kernel); other
# configs and kernels report null.
MEASURED_TRAFFIC = {
    ("c1", "k_sweep_win<B16P,float,6>"): 246316000,
}


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def sweep_bytes(nnzb, nnod, blk_val_bytes=72, vec_bytes=8, windows=0):
    """Algorithmic bytes of one fused Jacobi sweep r = r0 - K d; d' = d + w D^-1 r
    on the fine level: every stored 3x3 block once (its nine values,
    blk_val_bytes: 72 in FP64, 20 in the packed BF16 layout of eight BF16
    values and an FP32 v8; + its column: an int32, or a two-byte place in the
    window on a level that the context sweeps in windows), the row table, and per
    row the vectors d (gather, perfect reuse), r0, D^-1 read and d' written."""
    return nnzb * (blk_val_bytes + (2 if windows else 4)) + nnod * 4 + nnod * 3 * 4 * vec_bytes


def cpu_threads():
    """Threads for the CPU baseline: the cores this process may use, at most
    16 (one GPU's share of the host)."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(16, n))


def cpu_baseline(mesh, inp, Visc, Dens, start, opts, rel_res_fn, nthreads):
    """The complete solve on the host: the FP64 C++/OpenMP restatement of the
    same algorithm (oracle/cpu_stokes.cpp: assembly, Galerkin products,
    envelope Cholesky, Patera with MGPCG), on the same inputs, from the same
    starting point and with the same stopping rule as the timed GPU leg.
    Set-up (patterns, slot maps, orderings) is excluded, as for the GPU."""
    from oracle import cpu_solver as CS
    t0 = time.perf_counter()
    s = CS.CpuStokes(mesh, inp["ifix"], inp["vfix"], nthreads=nthreads)
    t_setup = time.perf_counter() - t0
    U0, P0 = start
    t0 = time.perf_counter()
    U, P, info = s.solve(Visc, Dens, inp["phys"], U0=U0, P0=P0, **opts)
    sec = time.perf_counter() - t0
    s.close()
    rr = rel_res_fn(U, P)
    return dict(value=round(1.0 / sec, 5), unit="solves/s", cores=nthreads, kind="port",
                sample=("one complete solve of the same workload on the host: FP64 C++/OpenMP restatement "
                        f"(oracle/cpu_stokes.cpp) on {nthreads} threads, same inputs, same start and same "
                        "fixed-residual stopping rule as the timed GPU leg; set-up excluded"),
                s_per_solve=round(sec, 3), rel_res=float(f"{rr[0]:.3e}"),
                iterations={k: info[k] for k in ("nitP", "nitU", "nitZ")},
                phases_s={k: round(info[k], 3) for k in ("t_assemble", "t_restrict", "t_factor", "t_solve")},
                setup_s=round(t_setup, 2), coarse_factor_entries=info["coarse_env"]), U, P


def roofline(ctx, mesh, api, run_once, form, config):
    """Average duration of the fine-level fused sweep over one solve, and the
    aggregate over every V-cycle kernel of that solve (HIP events that each
    launch records at its start and end on the solver's stream; algorithmic
    bytes per launch from the library)."""
    api.profile(ctx, True)
    run_once()
    pr = api.profile_read(ctx)
    api.profile(ctx, False)
    st = ctx.stats()
    nnzb, nnod, windows = st["nnzb"][0], mesh.nnod, st["windows"][0]
    if form == "fp64":
        nsw, tsw, bsw, bpl = pr["n_fp64"], pr["t_fp64"], pr["b_fp64"], sweep_bytes(nnzb, nnod, 72, 8, windows)
    else:
        nsw, tsw, bsw, bpl = pr["n_mixed"], pr["t_mixed"], pr["b_mixed"], sweep_bytes(nnzb, nnod, 20, 4, windows)
    if nsw and abs(bsw / nsw - bpl) > 1e-6 * bpl:
        raise SystemExit(f"bench.py: sweep bytes disagree with the library ({bsw / nsw} vs {bpl})")
    avg = tsw / max(nsw, 1)
    achieved = bpl / avg / 1e9
    log(f"sweep: {nsw} launches avg {avg * 1e6:.1f} us, {bpl / 1e6:.1f} MB -> {achieved:.0f} GB/s")
    t_all, b_all, n_all = tsw + pr["t_vcycle_other"], bsw + pr["b_vcycle_other"], nsw + pr["n_vcycle_other"]
    vc = b_all / t_all / 1e9
    log(f"V-cycle: {n_all} launches, {t_all * 1e3:.2f} ms, {b_all / 1e9:.2f} GB -> {vc:.0f} GB/s")
    kern = ("k_sweep_win" if windows else "k_sweep") + ("<double,double,6>" if form == "fp64" else "<B16P,float,6>")
    cp = round(api.copy_rate(1 << 30, 20), 1)   # plain copy kernel of 1 GiB, read + write bytes
    log(f"copy kernel: {cp:.0f} GB/s")
    return dict(bound="hbm", achieved=round(achieved, 1), peak=HBM_PEAK_GBS, unit="GB/s",
                frac=round(achieved / HBM_PEAK_GBS, 4), traffic=MEASURED_TRAFFIC.get((config, kern)),
                kernel=f"{kern}: fine-level fused Jacobi sweep", launches=nsw,
                avg_us=round(avg * 1e6, 2), bytes_per_launch=int(bpl),
                vcycle=dict(achieved=round(vc, 1), frac=round(vc / HBM_PEAK_GBS, 4), launches=n_all,
                            kernel_ms=round(t_all * 1e3, 3), bytes=int(b_all),
                            what="sum of algorithmic bytes / sum of kernel time over every V-cycle kernel "
                                 "of one solve (sweeps on all levels, transfers, coarse triangular solves)"),
                copy_peak_measured=cp)


def diffusion_bench(args):
    """One JSON line for the thermal diffusion step (see the module docstring)."""
    from m3tet_sph_amd import mesh as M, api

    t0 = time.perf_counter()
    m = M.build_config(args.config)
    if args.grid == "vertex":
        EL4, n = m.levels[0].EL2NOD[:, :4], m.nVnod
    else:
        EL4, _ = M.p2_to_p1(m.GCOORD, m.levels[0].EL2NOD)
        n = m.nnod
    X = m.GCOORD[:n]
    h_min = min(float(np.min(np.linalg.norm(X[EL4[:, i]] - X[EL4[:, j]], axis=1)))
                for i in range(4) for j in range(i + 1, 4))
    dt = 1.0
    kappa = h_min ** 2 / dt
    ctx = api.StokesContext(m)
    ctx.diffusion_mesh(EL4, n)
    T0 = np.random.default_rng(0).random(n)
    ifix = np.nonzero(np.isin(m.PointID[:n], (301, 306)))[0]
    vfix = np.where(m.PointID[ifix] == 301, 1.0, 0.0)
    log(f"setup {time.perf_counter() - t0:.1f}s {args.config} {args.grid}: {len(EL4)} tets, {n} nodes, "
        f"kappa {kappa:.3e}")
    for _ in range(args.warmup):
        ctx.diffusion3d(T0, kappa, dt, ifix, vfix)
    infos = []
    t = time.perf_counter()
    for _ in range(args.steps):
        T, info = ctx.diffusion3d(T0, kappa, dt, ifix, vfix)
        infos.append(info)
    sec = (time.perf_counter() - t) / args.steps
    pairs = np.concatenate([EL4[:, i].astype(np.int64) * n + EL4[:, j] for i in range(4) for j in range(4)])
    nnz = int(np.unique(pairs).size)
    del pairs
    out = {"metric": "thermal diffusion steps/s (assembly + Jacobi PCG to 1e-8), 1 GPU",
           "value": round(1.0 / sec, 3), "unit": "steps/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": round(1e3 * sec, 3), "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic",
           "config": {"workload": f"{args.config} {args.grid}: {len(EL4)} linear tetrahedra, {n} nodes, "
                                  f"kappa dt / h_min^2 = 1, random initial temperature"},
           "nit": infos[-1]["nit"],
           "t_assemble_ms": round(1e3 * float(np.mean([i["t_assemble"] for i in infos])), 3),
           "t_solve_ms": round(1e3 * float(np.mean([i["t_solve"] for i in infos])), 3),
           "nnz": nnz, "spmv_bytes": nnz * 12 + n * 16}
    if not args.no_cpu:
        from oracle import diffusion as OD
        t = time.perf_counter()
        To, io = OD.diffusion3d_p(T0, kappa, m.GCOORD, m.GCOORD_SPH, EL4, ifix, vfix, dt)
        tc = time.perf_counter() - t
        out["cpu_baseline"] = {"value": round(1.0 / tc, 4), "unit": "steps/s", "cores": 1, "kind": "port",
                               "sample": "the same step in the oracle (NumPy / SciPy, one process)",
                               "nit": io["nit"]}
        out["max_abs_diff_vs_oracle"] = float(np.abs(T - To).max())
    ctx.close()
    print(json.dumps(out), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--config", default="c1")
    ap.add_argument("--form", default="learned", choices=["learned", "fp64", "mixed"])
    ap.add_argument("--tol", type=float, default=1e-6)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--visc-contrast", type=float, default=None,
                    help="default per config: c0 1e3, c1 1e4, c2 1e5, c4 1e6")
    ap.add_argument("--rtol-U-first", type=float, default=4e-7,
                    help="initial velocity solve of the warm-started legs: stop at this fraction of |f_U| "
                         "(default 4e-7 = rtol_U * rtol_restart, the reference's factor, on the fixed "
                         "denominator like every other stage); 0 keeps the reference's tolerance relative "
                         "to the starting residual, which a better start only tightens")
    ap.add_argument("--path", default="stokes", choices=["stokes", "diffusion"])
    ap.add_argument("--grid", default="vertex", choices=["vertex", "p2split"])
    args = ap.parse_args()
    vc = args.visc_contrast or {"c0": 1e3, "c1": 1e4, "c2": 1e5, "c4": 1e6}.get(args.config, 1e4)
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py: this build runs on exactly one GPU (the Stokes solve is single-device; "
              "multi-GPU sharding is a design note only). Use --gpus 1.", file=sys.stderr)
        sys.exit(2)
    if args.path == "diffusion":
        diffusion_bench(args)
        return

    from m3tet_sph_amd import mesh as M, fields as F, api

    t0 = time.perf_counter()
    mesh = M.build_config(args.config)
    # c4 adds a Gaussian thermal plume (dT 0.3, radius 0.05) at the CMB (theta 0.9, phi 1.3)
    plume = (0.3, 0.05, 0.9, 1.3) if args.config == "c4" else None
    inp = F.make_inputs(mesh, visc_contrast=vc, Ra=1e5, seed_T=0, seed_plates=1, plume=plume)
    ctx = api.StokesContext(mesh)
    ctx.set_bc(inp["ifix"], inp["vfix"])
    phys = inp["phys"]
    log(f"setup {time.perf_counter() - t0:.1f}s config={args.config} nel={mesh.nel} "
        f"nU={3 * mesh.nnod} nP={mesh.nVnod} stats={ctx.stats()}")

    net = None
    workload = "seed-0 temperature field, cold start"
    if args.form == "learned":
        from m3tet_sph_amd import learned as L
        data = os.path.join(HERE, "m3tet_sph_amd", "data")
        wpath = os.path.join(data, f"warm_start_{args.config}.npz")
        spath = os.path.join(data, f"{args.config}_heldout_states.npz")
        if not (os.path.exists(wpath) and os.path.exists(spath)):
            raise SystemExit(f"bench.py: trained network or held-out states missing ({wpath}, {spath}); "
                             f"run python -m m3tet_sph_amd.train_warm_start first")
        net = L.WarmStartNet(mesh)
        meta = net.load(wpath)
        z = np.load(spath, allow_pickle=False)
        step, order = int(z["steps"][-1]), int(z["order"])
        if int(meta.get("order", -1)) != order:
            raise SystemExit(f"bench.py: {wpath} was trained with order {meta.get('order')}, states have {order}")
        T_hist, t_hist = z["T_hist"][-1], z["t_hist"][-1]
        Tv, t_k = T_hist[-1], float(t_hist[-1])
        net.clear_history()
        for T_j, t_j in zip(T_hist[:-1], t_hist[:-1]):
            # converged as a time loop converges them: to the same rel.res as the timed solves
            Vj, Dj = F.material(L.nodal_temperature(mesh, T_j, net.edge_parent), vc)
            U_prev, P_prev, _ = ctx.flow3d(Vj, Dj, phys, rtol_Pat=0.8 * args.tol, rtol_U_final=0.5 * args.tol)
            net.push_state(float(t_j), T_j, U_prev, P_prev)
        Visc, Dens = F.material(L.nodal_temperature(mesh, Tv, net.edge_parent), vc)
        workload = (f"held-out step {step} of the seeded convection trajectory (seed 2), "
                    f"converged states of steps {step - order - 1}..{step - 1} given")
    else:
        Visc, Dens = inp["Visc"], inp["Dens"]

    def cold(form):
        return ctx.flow3d(Visc, Dens, phys, P0=None, rtol_Pat=0.8 * args.tol, rtol_U_final=0.5 * args.tol,
                          precision=form)

    # fixed denominator: pressure residual of the velocity solve at P = 0
    U, P, info = cold("fp64")
    rP_cold = info["norm_rP0"]
    tol_abs = 0.8 * args.tol * rP_cold  # margin: the final velocity solve moves r_P slightly

    # The warm legs run device-resident, as a time loop that keeps its state
    # on the GPU would: the step's fields and the network's inputs are
    # uploaded before the timed region, every start is formed on the device
    # (order 0 of the pushed history is the previous step's state), and the
    # solution stays there (read back after the timed region).
    if net is not None:
        ctx.set_fields(Visc, Dens)
        net.set_inputs(Tv, Visc)
    wopts = dict(rtol_U_final=0.5 * args.tol, tol_Pat_abs=tol_abs, rtol_U_first=args.rtol_U_first)

    def from_device(form):  # the start that the network context holds on the GPU
        return ctx.flow3d(None, None, phys, start_device=net.start_device(), precision=form, keep_on_device=True,
                          **wopts)

    def prev(form):
        net.extrapolate(t_k, 0, device=True)
        return from_device(form)

    def extrap(form):
        net.extrapolate(t_k, order, device=True)
        return from_device(form)

    def learned(form):  # the network's start formed while the solve assembles and factorises
        return net.solve(ctx, t_k, order, phys, keep_on_device=True, precision=form, **wopts)

    def learned_host(form):  # the same solve through host buffers (fields in, solution out)
        net.warm_start_hist(t_k, order, Tv, Visc, device=True)
        return ctx.flow3d(Visc, Dens, phys, start_device=net.start_device(), precision=form, **wopts)

    def rel_res(U, P):
        rU, fU, rP = api.residual(ctx, U, P)
        return max(rU / fU, rP / rP_cold), rU / fU, rP / rP_cold

    def timed(fn):
        for _ in range(args.warmup):
            fn()
        t0 = time.perf_counter()
        infos = []
        for _ in range(args.steps):
            U, P, info = fn()
            infos.append(info)
        dt = time.perf_counter() - t0
        if U is None:  # device-resident solve: read the solution back after the timed region
            U, P = ctx.solution()
        rr = rel_res(U, P)
        res = dict(solves_per_s=round(args.steps / dt, 4), ms_per_solve=round(1e3 * dt / args.steps, 2),
                   rel_res=float(f"{rr[0]:.3e}"), nitP=infos[-1]["nitP"], nitU=infos[-1]["nitU"],
                   nitZ=infos[-1]["nitZ"])
        return res, U, P, infos

    legs = {}
    plain, Up, Pp, plain_infos = timed(lambda: cold("fp64"))
    log(f"plain fp64 (cold): {plain}")
    if args.form == "learned":
        legs["fp64_prev_step"], _, _, _ = timed(lambda: prev("fp64"))
        legs["mixed_prev_step"], _, _, _ = timed(lambda: prev("mixed"))
        legs["fp64_extrapolated"], _, _, _ = timed(lambda: extrap("fp64"))
        legs["mixed_extrapolated"], _, _, _ = timed(lambda: extrap("mixed"))
        legs["fp64_learned"], _, _, _ = timed(lambda: learned("fp64"))
        for k, v in legs.items():
            log(f"{k}: {v}")
        legs["mixed_learned_host_buffers"], _, _, _ = timed(lambda: learned_host("mixed"))
        main_fn, vform = (lambda: learned("mixed")), "mixed"
    elif args.form == "mixed":
        main_fn, vform = (lambda: cold("mixed")), "mixed"
    else:
        main_fn, vform = (lambda: cold("fp64")), "fp64"
    if args.form == "fp64":
        res, U, P, infos = plain, Up, Pp, plain_infos
    else:
        res, U, P, infos = timed(main_fn)
    ms = res["ms_per_solve"]
    rr, rru, rrp = rel_res(U, P)
    err_vs_fp64 = dict(U=float(f"{np.linalg.norm(U - Up) / np.linalg.norm(Up):.3e}"),
                       P=float(f"{np.linalg.norm(P - Pp) / np.linalg.norm(Pp):.3e}"))
    log(f"{args.form}: {res}; rel_res={rr:.2e} (U {rru:.2e}, P {rrp:.2e}); last info {infos[-1]}")

    roof = roofline(ctx, mesh, api, main_fn, vform, args.config)

    cpu = None
    if not args.no_cpu:
        # the timed leg's start, on the host: the network start (extrapolation +
        # correction) of the learned form, P = 0 and U from the BCs otherwise
        if args.form == "learned":
            start = net.warm_start_hist(t_k, order, Tv, Visc)
            copts = dict(rtol_U_final=0.5 * args.tol, tol_Pat_abs=tol_abs, rtol_U_first=args.rtol_U_first)
        else:
            start = (None, None)
            copts = dict(rtol_Pat=0.8 * args.tol, rtol_U_final=0.5 * args.tol)
        t0 = time.perf_counter()
        cpu, Uc, Pc = cpu_baseline(mesh, inp, Visc, Dens, start, copts, rel_res, cpu_threads())
        cpu["diff_vs_gpu"] = dict(U=float(f"{np.linalg.norm(Uc - U) / np.linalg.norm(U):.3e}"),
                                  P=float(f"{np.linalg.norm(Pc - P) / np.linalg.norm(P):.3e}"))
        log(f"cpu baseline took {time.perf_counter() - t0:.1f}s: {cpu}")

    last = infos[-1]
    out = {
        "metric": "Stokes solves/s to rel.res 1e-6: mixed+learned vs plain FP64 MGPCG, 1 GPU",
        "value": round(1e3 / ms, 4),
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 2),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if vform == "fp64" else "f64 outer, f32/bf16 V-cycle",
        "data": "synthetic",
        "config": {"workload": f"{args.config}: spherical-shell Stokes, {mesh.nel} P2 tets, "
                               f"{3 * mesh.nnod} velocity dofs, {mesh.nVnod} pressure dofs, "
                               f"{mesh.nmg}-level MG, viscosity contrast {vc:.0e}; {workload}",
                   "form": {"learned": "mixed+learned", "fp64": "plain fp64", "mixed": "mixed"}[args.form],
                   "rel_res_target": args.tol, "seeds": [0, 1, 2], "Ra": 1e5,
                   "residency": ("device: the step's fields, the network's inputs and the converged history "
                                 "in HBM before the timed region, start formed and solution left in HBM; "
                                 "legs.mixed_learned_host_buffers is the same solve with host fields in and "
                                 "host solution out" if args.form == "learned" else
                                 "host buffers: fields in, solution out (cold start)"),
                   "stopping": (f"fixed denominators (|f_U|, cold |r_P|): first velocity solve "
                                f"{args.rtol_U_first:g} |f_U|, Patera {0.8 * args.tol:g} |r_P cold|, final "
                                f"velocity {0.5 * args.tol:g} |f_U|" if args.rtol_U_first > 0 else
                                f"first velocity solve relative to its start (reference rule), Patera "
                                f"{0.8 * args.tol:g} |r_P cold|, final velocity {0.5 * args.tol:g} |f_U|")},
        "rel_res": float(f"{rr:.3e}"),
        "iterations": {"nitP": last["nitP"], "nitU": last["nitU"], "nitZ": last["nitZ"]},
        "phases_ms": {k: round(1e3 * last[k], 2) for k in
                      ("t_assemble", "t_restrict", "t_factor", "t_pressure", "t_velocity")},
        "roofline": roof,
        "cpu_baseline": cpu,
        "plain_fp64": plain,
        "speedup_vs_plain_fp64": round(plain["ms_per_solve"] / ms, 3),
        "error_vs_fp64": err_vs_fp64,
    }
    if legs:
        out["legs"] = legs
        out["speedup_vs_fp64_prev_step"] = round(legs["fp64_prev_step"]["ms_per_solve"] / ms, 3)
        out["speedup_vs_mixed_extrapolated"] = round(legs["mixed_extrapolated"]["ms_per_solve"] / ms, 3)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
