#!/usr/bin/env python3
"""Benchmark: Crank-Nicolson steps/s of the GaDE hot path on one MI355X.

Workload (default): non-dipole, Z=1, rBox=30, NSplines=250, NKappa=16, NMu=8,
Nl=8, 15-cycle sin^2 pulse, Omega=50, Intensity=10, dt = T/8000, BiCGSTAB
rel-tol 1e-12, psi0 = 1s ground state.  The state is first propagated (untimed)
to the middle of the pulse (--start-step, default Ntime/2, where the field and
the iteration counts are largest), then W warm-up steps, then K timed steps.  A "step" is one CN
step: f(t), rhs = (S - H) psi, preconditioned BiCGSTAB on (S + H) -- the
plain FP64 GPU form (fused operator, no assembly).  Inputs are generated by
dirac_hydrogen_code_amd.couplings (synthetic radial integrals, exact angular
couplings) and are resident in HBM before the timed region starts.

Prints ONE JSON line.  Only --gpus 1 is supported: the problem sits on one GPU.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "CN steps/s + BiCGSTAB iters/step, FP64 vs mixed+learned at ‖Δψ‖≤1e-8"
HBM_PEAK_GBS = 8000.0
FP64_PEAK_TFS = 78.6

WORKLOADS = {
    "nondipole_ns250_k16_mu8_l8": dict(ntime=8000, E0=10.0, omega=50.0, cycles=15.0, lmax=8),
    "dipole_ns50_k4_l1": dict(ntime=200, E0=10.0, omega=50.0, cycles=1.0, lmax=1),
}


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def advance(t, k, dt):
    """Time after k more steps, accumulated one dt at a time as the reference loop does
    (tools/dirac_solver.c:509)."""
    for _ in range(k):
        t = t + dt
    return t


def host_info():
    """CPU model, logical CPUs of the machine and CPUs this process may run on."""
    model = None
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
    return dict(cpu_model=model, nproc=os.cpu_count(), affinity=affinity)


def ensure_inputs(config, datadir):
    from dirac_hydrogen_code_amd.couplings import CONFIGS, generate
    marker = os.path.join(datadir, "params.json")
    if not os.path.exists(marker):
        log(f"generating inputs for {config} in {datadir}")
        t = time.time()
        generate(datadir, **CONFIGS[config])
        log(f"  generated in {time.time() - t:.1f}s")
    return datadir


def real_form(gp):
    """Whether the generated couplings and a real f(t) run the banded kernels' real form (zero quadrants left out)."""
    return gp.get_param("radial") == 2 and not gp.get_param("radial_mfma") and bool(gp.get_param("ang_list"))


def kernel_models(gp):
    """Algorithmic work per launch of each kernel family (flops or HBM bytes)."""
    from dirac_hydrogen_code_amd.couplings import csr_read
    nb, n, nnzb, L = gp.nblk, gp.blkdim, gp.nnz_b, gp.lmax
    N = gp.n
    # angular contraction: 2 complex MACs per (l, non-zero of H0l or H1l between kept blocks) per radial entry
    Hall = csr_read(os.path.join(gp.directory, "H.csr"))
    perm = Hall["perm"]
    rows = np.repeat(np.arange(Hall["n"]), np.diff(Hall["Ap"]))
    ang_nnz = 0
    for l in range(L):
        for nm in ("H0l", "H1l"):
            A = csr_read(os.path.join(gp.directory, f"{nm}{l}.csr"))
            from scipy import sparse
            D = sparse.csr_matrix((A["Ax"], A["Ai"], A["Ap"]), shape=(A["n"], A["n"]))
            vals = np.asarray(D[perm[rows], perm[Hall["Ai"]]]).ravel()
            ang_nnz += int(np.count_nonzero(vals))
    nnz_full = gp.hall_nnz * nnzb
    # the banded kernel runs the generated couplings on real coefficients (4 flops a product instead of 8) and leaves
    # out a quarter of the G products, zero in their basis; the stationary operator is complex
    real = real_form(gp)
    radial = nb * nnzb * ((12.0 if real else 32.0) * L + 8.0)
    # the fused form does the angular contraction inside the radial kernel, without the vanishing products' windows
    fused = gp.get_param("ang_fused") and gp.get_param("radial") == 2 and not gp.get_param("radial_mfma")
    angular = (16.0 if not real else 6.0 if fused else 8.0) * ang_nnz * n
    return {
        # fused radial SpMM: per block, 4 kappa-folded radial products per l + the diagonal operator (and the
        # angular contraction with ang_fused)
        "radial": dict(bound="mfma", flops=radial + (angular if fused else 0.0)),
        "angular": dict(bound="mfma", flops=angular),
        # equivalent assembled SpMV of S + Hfull (8 flops per non-zero of S + Hfull per A-apply)
        "aapply_equiv": dict(bound="mfma", flops=8.0 * (nnz_full + nb * nnzb)),
        "csr_spmv": dict(bound="hbm", bytes=nnz_full * 20.0 + (N + 1) * 4.0 + 2 * N * 16.0),
        "psolve": dict(bound="hbm", bytes=2.0 * N * 16.0),
        "blas1": dict(bound="hbm", bytes=4.0 * N * 16.0),
        # per-multipole partial outputs summed in a fixed order
        "radial_sum": dict(bound="hbm", bytes=(L + 1) * N * 16.0 + N * 16.0),
        "gsums": dict(bound="hbm", bytes=L * nnzb * (144.0 if real else 320.0)),
    }


# device kernels behind each timed family (the names rocprofv3 reports)
KERNEL_NAMES = {"radial": "k_radial_dia<7, false, double2>", "radial_pair": "k_radial_dia<7, true, double2>",
                "angular": "k_angular<4, double2>", "psolve": "k_psolve_tw<2, double2, 2, 1>", "gsums": "k_gsums_kb",
                "blas1": "k_bicg", "csr_spmv": "k_csr_spmv"}


def measured_traffic(workload, kernel):
    """HBM bytes per launch of 'kernel' from the committed FETCH_SIZE/WRITE_SIZE summary, or None.

    The summary holds the counters' KiB per dispatch and the factor that maps each
    counter onto the bytes a plain copy kernel of known size moves."""
    path = os.path.join(ROOT, "profiles", f"traffic_{workload}.json")
    if not kernel or not os.path.exists(path):
        return None
    with open(path) as f:
        t = json.load(f)
    ks = t.get("kernels", {})
    k = ks.get(kernel) or next((v for name, v in ks.items() if name.startswith(kernel + "<")), None)
    if not k:
        return None
    return 1024.0 * (k["fetch_kib"] * t["fetch_scale"] + k["write_kib"] * t["write_scale"])


def mixed_variant(args, gp, dpsi, psi_window, psi_fp64_end, wl, t_start):
    """The same window from the same psi in the mixed-precision form (FP32 inner BiCGSTAB and block-LU
    apply, FP64 defect correction to the same tolerance), after the same autotuning; its end state against
    the FP64 one, then a short pass with the FP32 kernel families timed."""
    from dirac_hydrogen_code_amd import gade
    lib = gade.lib()
    gp.set_param("precision", 1)
    dpsi.upload(psi_window)
    gp.reset_workspace()
    pr = [(wl["E0"], wl["omega"], wl["cycles"], 0.0)]
    chosen, rows = gp.autotune(dpsi, pr, args.tune or 16, t0=t_start, tol=args.tol, reps=2)
    gade.check(lib.gade_device_sync())
    w = time.perf_counter()
    it, tols, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.steps, t0=t_start, tol=args.tol,
                            timing=False)
    gade.check(lib.gade_device_sync())
    el = time.perf_counter() - w
    x = dpsi.get()
    err = float(np.linalg.norm(x - psi_fp64_end) / np.linalg.norm(psi_fp64_end))
    norm = gp.snorm(dpsi)
    # per-family times of the mixed step (launches the device loop gates off are left out)
    gp.set_param("profile_floor_ns", 20000)
    gp.profile("all")
    gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], 10, t0=t_start + args.steps * gp.dt, tol=args.tol,
              timing=False)
    fams = {}
    for name in ("angular", "radial_pair", "radial", "angular_f32", "radial_f32", "psolve_f32", "blas1_f32",
                 "radial_sum_f32", "radial_sum", "gsums"):
        tot, cnt = gp.profile_get(name)
        if cnt:
            fams[name] = dict(avg_us=1000.0 * tot / cnt, count=cnt)
    gp.profile(False)
    gp.set_param("profile_floor_ns", 0)
    gp.set_param("precision", 0)
    out = dict(value=args.steps / el, inner_iters_per_step=float(it.mean()), max_tol_error=float(tols.max()),
               final_rel_diff_vs_fp64=err, s_norm=norm, chosen=rows[chosen], kernels=fams,
               note="same window and psi; complex64 inner BiCGSTAB + block-LU apply, FP64 residual/update/"
                    "tolerance; iterations are inner iterations (every one counted)")
    log(f"mixed: {out['value']:.1f} steps/s, inner iters/step {it.mean():.2f}, |psi - psi_fp64|/|psi_fp64| "
        f"{err:.2e}, " + ", ".join(f"{k} {v['avg_us']:.1f}us" for k, v in fams.items()))
    return out


def learned_production(args, gp, dpsi, psi_window, psi_fp64_end, wl, datadir, t_start):
    """The learned guess at the production size: trained on a batched model of the same couplings with seeded
    pulses (0x5EED, disjoint from the timed pulse), installed into the single-instance model, then the timed
    window from the same psi with the extrapolated guess and with the learned guess in FP64 and in the
    mixed-precision form."""
    from dirac_hydrogen_code_amd import gade, learned
    lib = gade.lib()
    t0 = time.perf_counter()
    gt = gade.Propagator(datadir, wl["lmax"], gp.dt, batch=args.lg_prod_batch)
    gt.set_param("graph", 0 if args.no_graph else 1)
    psi0, _ = gade.read_psi0(datadir, gp.n)
    # the timed run is the reference's pulse (fixed carrier phase) at the middle of its envelope: train on that
    # pulse family, with seeded amplitudes, frequencies and lengths, short enough (2..4 cycles) that the steps
    # the samples cover run through each pulse's peak field
    tr = learned.Trainer(gt, psi0, seed=0x5EED, npod=args.lg_prod_npod, nsnap=400, nsamples=args.lg_prod_samples,
                         log=log, cep=0.0, ranges=dict(E0=(3.0, 30.0), omega=(40.0, 60.0), cycles=(2, 4)))
    tr.build_pod(snap_every=0)
    tr.collect_samples()
    _, v0, v1 = tr.fit(epochs=args.lg_epochs, M=256, lr=1e-3, lr_final=1e-4)
    tr.export_to(gp)
    t_train = time.perf_counter() - t0
    out = dict(train_seconds=t_train, train_instances=args.lg_prod_batch, train_samples=int(len(tr.valid)),
               zero_weight_samples=tr.nzero, validation_loss_before=v0, validation_loss_after=v1, forms={})
    del tr, gt
    for key, prec, go in (("fp64_extrapolation", 0, 2), ("fp64_learned", 0, gade.GUESS_LEARNED),
                          ("mixed_learned", 1, gade.GUESS_LEARNED)):
        gp.set_param("precision", prec)
        gp.set_param("guess_order", go)
        gp.set_param("lg_features", 0)
        # a warm-up call (first-use buffers, captures), for the learned forms the autotuner (its probes leave psi
        # and the solver state as they were; the extrapolated form, first, keeps the plain run's choice), then
        # the timed call from the same psi
        dpsi.upload(psi_window)
        gp.reset_workspace()
        gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], 8, t0=t_start, tol=args.tol, timing=False)
        dpsi.upload(psi_window)
        gp.reset_workspace()
        tuned = None
        if args.tune and go == gade.GUESS_LEARNED:
            ch, rows = gp.autotune(dpsi, [(wl["E0"], wl["omega"], wl["cycles"], 0.0)], args.tune, t0=t_start,
                                   tol=args.tol, reps=2)
            tuned = rows[ch]
        dpsi.upload(psi_window)
        gp.reset_workspace()
        gade.check(lib.gade_device_sync())
        w = time.perf_counter()
        it, tols, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.steps, t0=t_start, tol=args.tol,
                                timing=False)
        gade.check(lib.gade_device_sync())
        el = time.perf_counter() - w
        x = dpsi.get()
        err = float(np.linalg.norm(x - psi_fp64_end) / np.linalg.norm(psi_fp64_end))
        out["forms"][key] = dict(value=args.steps / el, iters_per_step=float(it.mean()), max_tol_error=float(tols.max()),
                                 rel_diff_vs_fp64_plain=err, autotuned=tuned)
        if go == gade.GUESS_LEARNED:
            net, gated = (int(v) for v in gp.lg_uses()[0])
            out["forms"][key].update(network_steps=net, range_gate_fallback_steps=gated)
            log(f"  {key}: network used on {net} steps, range gate (|z| > {gp.get_param('lg_zmax')}) sent {gated} "
                f"to the extrapolation")
        log(f"production {key}: {args.steps / el:.1f} steps/s, iters/step {it.mean():.3f}, "
            f"|psi - psi_fp64|/|psi_fp64| {err:.1e}")
    gp.set_param("precision", 0)
    gp.set_param("guess_order", 0)
    out["note"] = ("same window and psi as the timed region; iterations of the mixed form are inner iterations; "
                   "training: seeded pulses of the reference's pulse family (carrier phase fixed, E0, omega, cycles "
                   "seeded 0x5EED) on the production couplings, POD of 400 extrapolation-defect snapshots, "
                   "snapshot and sample solves at tolerance 1e-13")
    return out


def learned_scan(args):
    """Learned initial guess on the batched scan: trained on seeded pulses disjoint from the timed scan
    (snapshots, POD, samples and training on the device), then the timed scan's first steps with the plain,
    extrapolated and learned guesses, in FP64 and in the mixed-precision form."""
    from dirac_hydrogen_code_amd import gade, learned
    wl = WORKLOADS["dipole_ns50_k4_l1"]
    datadir = ensure_inputs("dipole_ns50_k4_l1", os.path.join("/tmp", "gade_data", "dipole_ns50_k4_l1"))
    dt = (wl["cycles"] * 2 * np.pi / wl["omega"]) / wl["ntime"]
    B = args.batch
    lib = gade.lib()
    gp = gade.Propagator(datadir, wl["lmax"], dt, batch=B)
    gp.set_param("graph", 0 if args.no_graph else 1)
    psi0, _ = gade.read_psi0(datadir, gp.n)
    t0 = time.perf_counter()
    tr = learned.Trainer(gp, psi0, seed=0x5EED, nsnap=400, nsamples=args.lg_samples, log=log)
    tr.build_pod()
    tr.collect_samples()
    hist, v0, v1 = tr.fit(epochs=args.lg_epochs, M=256, lr=1e-3, lr_final=1e-4)
    t_train = time.perf_counter() - t0
    params, nsteps_b = learned.scan_pulses(0x6ADE, B, dt)
    K = min(args.batch_steps, int(nsteps_b.min()))
    out = dict(train_seconds=t_train, train_samples=int(len(tr.valid)), validation_loss_before=v0,
               validation_loss_after=v1, steps=K, forms={})
    ref = None
    for prec in (0, 1):
        gp.set_param("precision", prec)
        for name, go in (("plain", 0), ("extrapolation", 2), ("learned", gade.GUESS_LEARNED)):
            gp.set_param("lg_features", 0)
            gp.set_param("guess_order", go)
            x = gade.DeviceArray.from_host(np.tile(psi0, B))
            gp.reset_workspace()
            gp.cn_run_batch(x, params, 3, nsteps_b=nsteps_b)  # warm-up (graph capture, first launches)
            x.upload(np.tile(psi0, B))
            gp.reset_workspace()
            gade.check(lib.gade_device_sync())
            t = time.perf_counter()
            it, tols = gp.cn_run_batch(x, params, K, nsteps_b=nsteps_b)
            gade.check(lib.gade_device_sync())
            el = time.perf_counter() - t
            xs = x.get()
            if ref is None:
                ref = xs
            diff = float(np.linalg.norm(xs - ref) / np.linalg.norm(ref))
            key = ("fp64" if prec == 0 else "mixed") + "_" + name
            out["forms"][key] = dict(value=B * K / el, iters_per_step=float(it.mean()), max_tol_error=float(tols.max()),
                                     rel_diff_vs_fp64_plain=diff)
            log(f"learned scan {key}: {B * K / el:.0f} instance-steps/s, iters/step {it.mean():.3f}, "
                f"|psi - psi_fp64_plain|/|psi_fp64_plain| {diff:.1e}")
    gp.set_param("precision", 0)
    gp.set_param("guess_order", 0)
    f = out["forms"]
    out["speedup_mixed_learned_vs_fp64_plain"] = f["mixed_learned"]["value"] / f["fp64_plain"]["value"]
    out["speedup_fp64_learned_vs_fp64_plain"] = f["fp64_learned"]["value"] / f["fp64_plain"]["value"]
    out["note"] = ("dipole NSplines 50 NKappa 4 Nl 1, B instances; trained on seeded pulses 0x5EED (POD of 400 "
                   "extrapolation-defect snapshots, samples of the quadratic guess-error form), timed on the 0x6ADE "
                   "scan; iterations of the mixed form are inner iterations")
    return out


def batch_scan(args, workload="dipole_ns50_k4_l1", B=None, K=None, tune_steps=16, reps=2):
    """Batched pulse scan: B instances sharing one workload's couplings, each with its own seeded pulse (E0
    log-uniform in [1,100], omega uniform in [25,75], carrier phase uniform in [0, 2 pi), cycles uniform in
    1..15), the workload's dt, per-instance step counts ceil(T_i/dt).  Times the first K steps of the scan
    (every instance is still inside its pulse there) and, for comparison, the same steps of the first 4
    instances run one at a time."""
    from dirac_hydrogen_code_amd import gade
    wl = WORKLOADS[workload]
    datadir = ensure_inputs(workload, os.path.join("/tmp", "gade_data", workload))
    dt = (wl["cycles"] * 2 * np.pi / wl["omega"]) / wl["ntime"]
    rng = np.random.default_rng(0x6ADE)
    B = B or args.batch
    K = K or args.batch_steps
    E0 = np.exp(rng.uniform(np.log(1.0), np.log(100.0), B))
    om = rng.uniform(25.0, 75.0, B)
    cep = rng.uniform(0.0, 2 * np.pi, B)
    cyc = rng.integers(1, 16, B).astype(float)
    params = np.stack([E0, om, cyc, cep], axis=1)
    nsteps_b = np.ceil(cyc * 2 * np.pi / om / dt).astype(np.int32)
    K = min(K, int(nsteps_b.min()))
    gp = gade.Propagator(datadir, wl["lmax"], dt, batch=B)
    gp.set_param("graph", 0 if args.no_graph else 1)
    psi0, _ = gade.read_psi0(datadir, gp.n)
    x = gade.DeviceArray.from_host(np.tile(psi0, B))
    gp.cn_run_batch(x, params, 5, nsteps_b=nsteps_b)  # warm-up: builds the preconditioner, first launches
    x.upload(np.tile(psi0, B))
    gp.reset_workspace()
    # stepping parameters (window, iterations per enqueue, graph, kernel tiles) by the autotuner on the first
    # tune_steps steps
    chosen, rows = gp.autotune(x, params, tune_steps, reps=reps)
    tuned = rows[chosen]
    log(f"batch scan {workload} B={B} autotune: {tuned} of {len(rows)} candidates")
    lib = gade.lib()
    gade.check(lib.gade_device_sync())
    t = time.perf_counter()
    it, tols = gp.cn_run_batch(x, params, K, nsteps_b=nsteps_b)
    gade.check(lib.gade_device_sync())
    el = time.perf_counter() - t
    # the same steps one instance at a time (first 4 instances)
    g1 = gade.Propagator(datadir, wl["lmax"], dt, batch=1)
    g1.set_param("graph", 0 if args.no_graph else 1)
    ones = []
    for b in range(min(4, B)):
        y = gade.DeviceArray.from_host(psi0)
        g1.reset_workspace()
        g1.cn_run_batch(y, params[b:b + 1], 5)
        y.upload(psi0)
        g1.reset_workspace()
        gade.check(lib.gade_device_sync())
        t1 = time.perf_counter()
        g1.cn_run_batch(y, params[b:b + 1], K)
        gade.check(lib.gade_device_sync())
        ones.append(time.perf_counter() - t1)
    single = K / float(np.mean(ones))
    x_fp64 = x.get()
    # the same scan in the mixed-precision form
    mixed = None
    if args.mixed:
        gp.set_param("precision", 1)
        x.upload(np.tile(psi0, B))
        gp.reset_workspace()
        ch_m, rows_m = gp.autotune(x, params, tune_steps, reps=reps)
        gade.check(lib.gade_device_sync())
        t = time.perf_counter()
        it_m, tols_m = gp.cn_run_batch(x, params, K, nsteps_b=nsteps_b)
        gade.check(lib.gade_device_sync())
        el_m = time.perf_counter() - t
        xm = x.get().reshape(B, -1)
        xf = x_fp64.reshape(B, -1)
        errs = np.linalg.norm(xm - xf, axis=1) / np.linalg.norm(xf, axis=1)
        mixed = dict(value=B * K / el_m, inner_iters_per_step=float(it_m.mean()),
                     max_tol_error=float(tols_m.max()), max_rel_diff_vs_fp64=float(errs.max()),
                     autotuned=rows_m[ch_m])
        gp.set_param("precision", 0)
        log(f"batch scan mixed: {mixed['value']:.0f} instance-steps/s, inner iters/step {it_m.mean():.2f}, "
            f"max |psi - psi_fp64|/|psi_fp64| {errs.max():.2e}")
    out = dict(value=B * K / el, unit="instance CN steps/s", batch=B, steps=K, seconds=el,
               iters_per_step=float(it.mean()), max_tol_error=float(tols.max()),
               single_instance_steps_per_s=single, speedup_vs_one_at_a_time=B * K / el / single,
               autotuned=tuned, mixed=mixed,
               note=f"{workload} couplings shared by all instances; seeded pulses (0x6ADE)")
    log(f"batch scan {workload} B={B}: {out['value']:.0f} instance-steps/s over {K} steps ({el:.3f}s), one at a "
        f"time {single:.0f} steps/s -> x{out['speedup_vs_one_at_a_time']:.1f}")
    return out


def cpu_baseline(datadir, wl, dt, psi, t0, first_step, nsteps, threads, tol, how, all_cores=False, model=None):
    """The oracle (C restatement of the reference CPU path) on a bounded sample of the same workload:
    nsteps steps of the GPU's timed window from the GPU's psi at their start (how: which steps).
    Reference-faithful threading: OpenMP in the per-step assembly only; all_cores: the SpMV rows and the
    preconditioner blocks on the same threads too (same results).  Returns (result, x, model)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    tl = time.time()
    m = model or O.Model(datadir, wl["lmax"], dt, nthreads=threads)
    O.lib().or_model_set_threads(m.ptr, threads, 1 if all_cores else 0)
    m.reset_workspace()  # both samples start from a fresh BiCGSTAB workspace
    m.precond()
    log(f"  oracle ready in {time.time() - tl:.1f}s")
    t1 = time.time()
    x, iters, tols, usec = m.cn_run(psi, wl["E0"], wl["omega"], wl["cycles"], nsteps, t0=t0, tol=tol)
    el = time.time() - t1
    threading = (f"OpenMP ({threads} threads) in the per-step assembly, SpMV rows and preconditioner blocks "
                 f"(all-cores variant)" if all_cores else
                 f"OpenMP ({threads} threads) in the per-step assembly only, serial SpMV/LU/BiCGSTAB as the reference")
    return dict(value=nsteps / el, unit="CN steps/s", cores=threads, kind="port",
                sample=f"steps {first_step}..{first_step + nsteps - 1} ({how}) on the host CPU; {threading}; "
                       f"{el:.1f}s, mean {iters.mean():.2f} iters/step", host=host_info()), x, m


def main():
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--start-step", type=int, default=-1,
                    help="untimed CN steps from psi0 before the warm-up (-1: Ntime/2, the middle of the pulse)")
    ap.add_argument("--first-window", type=int, default=500,
                    help="also time steps 1..N from psi0 (the pulse onset; 0: skip)")
    ap.add_argument("--workload", default="nondipole_ns250_k16_mu8_l8", choices=sorted(WORKLOADS))
    ap.add_argument("--data", default=None, help="input directory (generated when missing)")
    ap.add_argument("--tol", type=float, default=1e-12)
    ap.add_argument("--profile-steps", type=int, default=3)
    ap.add_argument("--profile-period", type=int, default=7,
                    help="in the timed region, time every n-th launch of the dominant kernel")
    ap.add_argument("--cpu-steps", type=int, default=10, help="steps of the CPU baseline sample")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-spmv", action="store_true", help="skip the assembled-CSR SpMV measurement")
    ap.add_argument("--spmv-reps", type=int, default=20)
    ap.add_argument("--batch", type=int, default=64, help="also time the batched pulse scan with this many "
                    "instances on the dipole problem (0: skip)")
    ap.add_argument("--batch-steps", type=int, default=100)
    ap.add_argument("--prod-batch", type=int, default=64,
                    help="also time the batched pulse scan on the timed workload's couplings (0: skip)")
    ap.add_argument("--prod-batch-steps", type=int, default=20)
    ap.add_argument("--guess-variant", type=int, default=2,
                    help="also time the window with this extrapolation order of the initial guess (0: skip)")
    ap.add_argument("--tile-r", type=int, default=2, help="radial tile width (row blocks per tile)")
    ap.add_argument("--tune", type=int, default=16, help="autotuner probe steps before the timed region (0: defaults)")
    ap.add_argument("--unprofiled", type=int, default=1, help="rerun the window without event timing (0: skip)")
    ap.add_argument("--dia-rows", type=int, default=0, help="banded radial rows per tile (overrides tuning)")
    ap.add_argument("--dia-outputs", type=int, default=0, help="banded radial outputs per lane (overrides tuning)")
    ap.add_argument("--radial-mfma", type=int, default=-1,
                    help="1: FP64 radial products on the matrix cores, 0: vector units (-1: the library's default)")
    ap.add_argument("--ang-fused", type=int, default=-1,
                    help="1: the fused angular + radial form, 0: two kernels (overrides tuning; -1: tuned)")
    ap.add_argument("--dia-halves", type=int, default=0,
                    help="banded radial output halves per workgroup, 1 or 2 (overrides tuning)")
    ap.add_argument("--ang-lb", type=int, default=0, help="angular multipoles per block (overrides tuning)")
    ap.add_argument("--psolve-chunk", type=int, default=0, help="preconditioner level height, 16 or 32 (0: default)")
    ap.add_argument("--mixed", type=int, default=1, help="mixed-precision variants (0: skip)")
    ap.add_argument("--no-graph", action="store_true", help="no step graphs (e.g. under a kernel-trace profiler)")
    ap.add_argument("--lg-samples", type=int, default=20000, help="training samples of the learned guess (0: skip)")
    ap.add_argument("--lg-epochs", type=int, default=30, help="training epochs of the learned guess")
    ap.add_argument("--lg-prod-samples", type=int, default=20000,
                    help="training samples of the production-size learned guess (0: skip)")
    ap.add_argument("--lg-prod-batch", type=int, default=16, help="training pulses of the production-size learned guess")
    ap.add_argument("--lg-prod-npod", type=int, default=64, help="POD basis size of the production-size learned guess")
    ap.add_argument("--copy-probe-mb", type=int, default=256,
                    help="one device-to-device copy of this size before the run, the calibration kernel for "
                         "FETCH_SIZE/WRITE_SIZE counters")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build runs the whole problem on one GPU; --gpus must be 1 "
              "(multi-GPU sharding is a design note, not a measured path)", file=sys.stderr)
        sys.exit(2)

    from dirac_hydrogen_code_amd import gade
    wl = WORKLOADS[args.workload]
    datadir = ensure_inputs(args.workload, args.data or os.path.join("/tmp", "gade_data", args.workload))
    T = wl["cycles"] * 2 * np.pi / wl["omega"]
    dt = T / wl["ntime"]

    t0 = time.time()
    gp = gade.Propagator(datadir, wl["lmax"], dt)
    gp.set_param("graph", 0 if args.no_graph else 1)
    if args.radial_mfma >= 0:
        gp.set_param("radial_mfma", args.radial_mfma)
    psi, _ = gade.read_psi0(datadir, gp.n)
    dpsi = gade.DeviceArray.from_host(psi)
    lib = gade.lib()
    gade.check(lib.gade_precond_setup(gp.ptr))
    if args.tile_r:
        gp.set_param("tile_r", args.tile_r)
    log(f"model on device in {time.time() - t0:.1f}s: nblk={gp.nblk} blkdim={gp.blkdim} hall_nnz={gp.hall_nnz} "
        f"nnz_b={gp.nnz_b} nnz_full={gp.nnz_full} nkappa={gp.nkappa}")

    if args.copy_probe_mb:
        nb = args.copy_probe_mb << 20
        src, dst = gade.DeviceArray(nb // 16), gade.DeviceArray(nb // 16)
        gade.check(lib.gade_memcpy_d2d(dst.ptr, src.ptr, nb))
        gade.check(lib.gade_device_sync())
        src.free()
        dst.free()

    # propagate (untimed) to the start of the window: by default the middle of the pulse, where the field,
    # and with it the BiCGSTAB iteration count, is largest
    start = wl["ntime"] // 2 if args.start_step < 0 else args.start_step
    if start:
        t1 = time.time()
        gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], start, t0=0.0, tol=args.tol, timing=False)
        log(f"propagated to step {start} of {wl['ntime']} in {time.time() - t1:.1f}s")
    t_start = advance(0.0, start, dt)
    # warmup: W steps, then a short pass with every kernel family timed
    it_w, _, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.warmup, t0=t_start, tol=args.tol,
                           timing=False)
    t_start = advance(t_start, args.warmup, dt)
    fams = {}
    if args.profile_steps:
        # per-family breakdown with the host-driven loop: every launch is real work there
        gp.set_param("device_loop", 0)
        gp.profile("all")
        gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.profile_steps, t0=t_start, tol=args.tol,
                  timing=False)
        for name in gade.PROF:
            tot, cnt = gp.profile_get(name)
            if cnt:
                fams[name] = dict(total_ms=tot, count=cnt, avg_us=1000.0 * tot / cnt)
        gp.profile(False)
        gp.set_param("device_loop", 1)
        t_start = advance(t_start, args.profile_steps, dt)
        log("kernel families: " + ", ".join(f"{k} {v['avg_us']:.1f}us x{v['count']}" for k, v in fams.items()))
    dom = max(fams, key=lambda k: fams[k]["total_ms"]) if fams else "radial"

    psi_window = dpsi.get()  # start of the timed window, for the CPU sample and the variants
    first = start + args.warmup + args.profile_steps + 1  # number of the window's first step

    # kernel shapes and stepping picked by the autotuner on probe steps of this window (every candidate
    # gives the same trajectory bit for bit, and the solver state is restored, so the timed work is unchanged)
    tuned = None
    if args.tune:
        pr = [(wl["E0"], wl["omega"], wl["cycles"], 0.0)]
        chosen, rows = gp.autotune(dpsi, pr, args.tune, t0=t_start, tol=args.tol, reps=2)
        nshape = len(rows) - 40  # shape candidates first, then 40 stepping candidates
        radial = "mfma" if gp.get_param("radial_mfma") else "{dia_rows}x{dia_outputs} halves {dia_halves}"
        tuned = dict(chosen=rows[chosen], candidates=len(rows),
                     kernel_shapes_ms={(f"fused {radial.format(**r)}" if r["ang_fused"] else
                                        f"radial {radial.format(**r)} angular {r['ang_lb']}"): r["ms"]
                                       for r in rows[:nshape]})
        log(f"autotuned: {rows[chosen]} of {len(rows)} candidates")
    if args.dia_rows:
        gp.set_param("dia_outputs", 1)  # (rows, 1) is valid for every row count: the way to any other shape
    if args.ang_fused >= 0:
        gp.set_param("ang_fused", 0)  # set again below, after the tile shape it needs
    for name, val in (("dia_rows", args.dia_rows), ("dia_outputs", args.dia_outputs or (2 if args.dia_rows else 0)),
                      ("ang_lb", args.ang_lb), ("psolve_chunk", args.psolve_chunk), ("dia_halves", args.dia_halves)):
        if val:
            gp.set_param(name, val)  # explicit kernel shapes (e.g. to profile the tuned kernels without tuning)
    if args.ang_fused >= 0:
        gp.set_param("ang_fused", args.ang_fused)
    if gp.get_param("radial_mfma"):
        KERNEL_NAMES["radial"], KERNEL_NAMES["radial_pair"] = "k_radial_mfma<false, 8>", "k_radial_mfma<true, 8>"
    else:
        fused = gp.get_param("ang_fused")
        rp = f"{gp.get_param('dia_rows')}, {gp.get_param('dia_outputs')}"
        real = "true" if real_form(gp) else "false"
        form = f"{rp}, {gp.get_param('dia_halves')}, {'true' if fused else 'false'}, {real}, {real}>"
        KERNEL_NAMES["radial"] = f"k_radial_dia<7, false, double2, {form}"
        KERNEL_NAMES["radial_pair"] = f"k_radial_dia<7, true, double2, {form}"
    lb = f"{gp.get_param('ang_lb')}, double2"
    KERNEL_NAMES["angular"] = (f"k_angular_list<{lb}, {'true' if real_form(gp) else 'false'}>"
                               if gp.get_param("ang_list") else f"k_angular<{lb}>")

    # timed region: K steps continuing the trajectory; every profile_period-th launch of the dominant
    # family carries a HIP event pair (each pair costs a few microseconds of idle time on the stream);
    # launches that the device-driven loop gates off (they return within microseconds) are left out
    gp.set_param("profile_period", args.profile_period)
    gp.set_param("profile_floor_ns", 20000)  # gated launches return at once (under 10 us with their events)
    gp.profile([dom])
    gade.check(lib.gade_device_sync())
    w0 = time.perf_counter()
    iters, tols, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.steps, t0=t_start, tol=args.tol,
                               timing=False)
    gade.check(lib.gade_device_sync())
    elapsed = time.perf_counter() - w0
    dom_ms, dom_cnt = gp.profile_get(dom)
    gp.profile(False)
    gp.set_param("profile_period", 1)
    gp.set_param("profile_floor_ns", 0)
    steps_per_s = args.steps / elapsed
    norm = gp.snorm(dpsi)
    # populations of the window's end state by projection on the field-free eigenstates (per kappa)
    pops = gp.populations(dpsi)
    pops = dict(s_norm=pops["norm"], bound=pops["bound"], ionised=pops["ionised"],
                at_step=first + args.steps - 1)
    log(f"populations at step {pops['at_step']}: bound {pops['bound']:.12f}, ionised {pops['ionised']:.3e}, "
        f"S-norm {pops['s_norm']:.15f}")
    log(f"timed {args.steps} steps in {elapsed:.3f}s -> {steps_per_s:.1f} steps/s, iters/step {iters.mean():.2f}, "
        f"max tol {tols.max():.2e}, S-norm {norm:.15f}; {dom}: {dom_cnt} launches, "
        f"{1000.0 * dom_ms / max(dom_cnt, 1):.1f}us avg")

    models = kernel_models(gp)
    md = models[dom]
    avg_s = dom_ms / max(dom_cnt, 1) * 1e-3
    traffic = measured_traffic(args.workload, KERNEL_NAMES.get(dom))
    if md["bound"] == "hbm":
        ach = md["bytes"] / avg_s / 1e9
        roof = dict(bound="hbm", achieved=ach, peak=HBM_PEAK_GBS, unit="GB/s", frac=ach / HBM_PEAK_GBS,
                    traffic=traffic, kernel=dom, avg_us=avg_s * 1e6, launches=dom_cnt,
                    algorithmic_bytes=md["bytes"])
    else:
        ach = md["flops"] / avg_s / 1e12
        roof = dict(bound="mfma", achieved=ach, peak=FP64_PEAK_TFS, unit="TFLOP/s", frac=ach / FP64_PEAK_TFS,
                    traffic=traffic, kernel=dom, avg_us=avg_s * 1e6, launches=dom_cnt,
                    algorithmic_flops=md["flops"])

    variants = {}
    if args.guess_variant:
        # same window from the same psi with the extrapolated initial guess (history rebuilt inside the window)
        dpsi.upload(psi_window)
        gp.reset_workspace()
        gp.set_param("guess_order", args.guess_variant)
        gade.check(lib.gade_device_sync())
        w1 = time.perf_counter()
        it_g, tol_g, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.steps, t0=t_start,
                                   tol=args.tol, timing=False)
        gade.check(lib.gade_device_sync())
        el_g = time.perf_counter() - w1
        gp.set_param("guess_order", 0)
        variants[f"guess_order_{args.guess_variant}"] = dict(
            value=args.steps / el_g, iters_per_step=float(it_g.mean()), max_tol_error=float(tol_g.max()),
            note="same window and psi, x0 by polynomial extrapolation of the previous solutions")
        log(f"guess order {args.guess_variant}: {args.steps / el_g:.1f} steps/s, iters/step {it_g.mean():.2f}")

    if args.first_window:
        # steps 1..N from psi0 with the same tuned parameters: the pulse onset, where the field is weak
        psi0_h, _ = gade.read_psi0(datadir, gp.n)
        d0 = gade.DeviceArray.from_host(psi0_h)
        gp.reset_workspace()
        gade.check(lib.gade_device_sync())
        w3 = time.perf_counter()
        it_f, tol_f, _ = gp.cn_run(d0, wl["E0"], wl["omega"], wl["cycles"], args.first_window, t0=0.0,
                                   tol=args.tol, timing=False)
        gade.check(lib.gade_device_sync())
        el_f = time.perf_counter() - w3
        d0.free()
        variants["first_window"] = dict(value=args.first_window / el_f, iters_per_step=float(it_f.mean()),
                                        max_tol_error=float(tol_f.max()),
                                        note=f"steps 1..{args.first_window} from psi0 (pulse onset), same tuning")
        log(f"first window (steps 1..{args.first_window}): {args.first_window / el_f:.1f} steps/s, "
            f"iters/step {it_f.mean():.3f}")

    if args.unprofiled:
        # the same window and psi (workspace reset) with the same parameters, without kernel event timing
        # (the step graph may replay): what the event pairs of the timed region cost
        dpsi.upload(psi_window)
        gp.reset_workspace()
        gade.check(lib.gade_device_sync())
        w2 = time.perf_counter()
        it_a, tol_a, _ = gp.cn_run(dpsi, wl["E0"], wl["omega"], wl["cycles"], args.steps, t0=t_start,
                                   tol=args.tol, timing=False)
        gade.check(lib.gade_device_sync())
        el_a = time.perf_counter() - w2
        variants["no_event_timing"] = dict(value=args.steps / el_a, iters_per_step=float(it_a.mean()),
                                           max_tol_error=float(tol_a.max()),
                                           note="same window, psi and tuned parameters, no kernel event timing")
        log(f"no event timing: {args.steps / el_a:.1f} steps/s")
        psi_fp64_end = dpsi.get()

        if args.mixed:
            variants["mixed"] = mixed_variant(args, gp, dpsi, psi_window, psi_fp64_end, wl, t_start)
        if args.lg_prod_samples:
            variants["learned_production"] = learned_production(args, gp, dpsi, psi_window, psi_fp64_end, wl,
                                                                datadir, t_start)

    if args.prod_batch:
        # the same scan on the production couplings: every coupling read serves all instances of a step
        variants["batch_scan_production"] = batch_scan(args, args.workload, B=args.prod_batch,
                                                       K=args.prod_batch_steps, tune_steps=4, reps=1)
    if args.batch:
        variants["batch_scan"] = batch_scan(args)
        if args.lg_samples:
            variants["learned_scan"] = learned_scan(args)

    spmv = None
    if not args.no_spmv and args.spmv_reps > 0:
        # the reference's formulation on the same device: assembled Hfull (S excluded) and its CSR SpMV
        gp.set_time(gade.pulse(wl["E0"], wl["omega"], wl["cycles"], t_start))
        gp.profile(["assemble", "csr_spmv"])
        gp.assembled_timedep()
        dy = gade.DeviceArray(gp.n)
        for _ in range(args.spmv_reps):
            gp.assembled_spmv(dpsi, dy, alpha=1.0, beta=0.0, with_S=False)
        sp_ms, sp_cnt = gp.profile_get("csr_spmv")
        as_ms, as_cnt = gp.profile_get("assemble")
        gp.profile(False)
        sp_s = sp_ms / sp_cnt * 1e-3
        b = models["csr_spmv"]["bytes"]
        spmv = dict(kernel="k_csr_spmv", nnz=gp.nnz_full, avg_us=sp_s * 1e6, launches=sp_cnt,
                    algorithmic_bytes=b, achieved=b / sp_s / 1e9, peak=HBM_PEAK_GBS, unit="GB/s",
                    frac=b / sp_s / 1e9 / HBM_PEAK_GBS,
                    traffic=measured_traffic(args.workload, "k_csr_spmv"),
                    assemble_us=as_ms / max(as_cnt, 1) * 1e3)
        log(f"assembled SpMV: {spmv['avg_us']:.1f}us, {spmv['achieved']:.0f} GB/s ({100 * spmv['frac']:.1f}% of peak); "
            f"assembly {spmv['assemble_us']:.1f}us")
        dy.free()

    cpu = None
    if not args.no_cpu:
        hi = host_info()
        threads = min(16, hi["affinity"] or os.cpu_count() or 1)
        log(f"cpu baseline: {args.cpu_steps} step(s) with {threads} threads on {hi}")
        try:
            # a representative sample: the cpu_steps consecutive steps of the timed window whose GPU iteration
            # count is closest to the window's mean, started from the GPU's psi there
            k = min(args.cpu_steps, args.steps)
            run_mean = np.convolve(np.asarray(iters, float), np.ones(k), "valid") / k
            s0 = int(np.argmin(np.abs(run_mean - iters.mean())))
            for name, v in (("guess_order", 0), ("precision", 0)):
                gp.set_param(name, v)
            gp.reset_workspace()
            dps = gade.DeviceArray.from_host(psi_window)
            t_s = t_start
            if s0:
                gp.cn_run(dps, wl["E0"], wl["omega"], wl["cycles"], s0, t0=t_start, tol=args.tol, timing=False)
                t_s = advance(t_s, s0, dt)
            how = (f"the {k} consecutive steps of the timed window whose GPU iterations/step, {run_mean[s0]:.2f}, "
                   f"are closest to the window's {iters.mean():.3f}; from the GPU's psi there")
            psi_s = dps.get()
            cpu, _, om = cpu_baseline(datadir, wl, dt, psi_s, t_s, first + s0, k, threads, args.tol, how)
            # all cores of this process's share of the host (same sample, same results)
            allc = hi["affinity"] or os.cpu_count() or 1
            cpu_all, _, _ = cpu_baseline(datadir, wl, dt, psi_s, t_s, first + s0, k, allc, args.tol, how,
                                         all_cores=True, model=om)
            cpu["all_cores"] = dict(value=cpu_all["value"], cores=allc, sample=cpu_all["sample"])
            log(f"cpu baseline: {cpu['value']:.3f} steps/s reference-faithful ({threads} threads in the assembly), "
                f"{cpu_all['value']:.3f} steps/s on {allc} cores")
            del om
        except Exception as e:  # report, do not hide the GPU number
            log(f"cpu baseline failed: {e}")

    out = {
        "metric": METRIC,
        "value": steps_per_s,
        "unit": "CN steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1000.0 * elapsed / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic: generated coupling files of this shape (exact angular couplings, B-spline DKB-style radial integrals)",
        "config": {"workload": f"{args.workload} plain FP64 CN (fused operator)", "nblk": gp.nblk,
                   "blkdim": gp.blkdim, "lmax": gp.lmax, "dt": dt, "tol": args.tol,
                   "window": f"steps {first}..{first + args.steps - 1} of {wl['ntime']} (untimed propagation to "
                             f"step {start}, {args.warmup} warm-up and {args.profile_steps} profiled steps before)"},
        "iters_per_step": float(iters.mean()),
        "max_tol_error": float(tols.max()),
        "s_norm": norm,
        "populations": pops,
        "roofline": roof,
        "kernels": fams,
        "cpu_baseline": cpu,
        "assembled_spmv": spmv,
        "tuning": tuned,
        "variants": variants,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
