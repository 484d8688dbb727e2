#!/usr/bin/env python3
"""Benchmark: FP64 CSR SpMV + Jacobi-PCG on one MI355X.

Workload (the configuration the metric is quoted on), two inputs:
  (a) 3D 7-point Poisson, 192^3 grid: 7,077,888 rows, 49,324,032 nnz,
      Dirichlet diagonal 6;
  (b) power-law SPD, 4,194,304 rows: Zipf(1.5) row lengths on [3, 4096],
      symmetrised, values uniform[-1,0), diagonal = sum|off| + 1;
both with int32 indices, RHS splitmix64(seed 42) uniform[-1,1], x0 = 0,
relative residual tolerance 1e-8, Jacobi left preconditioner, plain PCG
(restart_iterations = max_iterations).  One step = one full PCG solve to 1e-8
of each input, matrices and vectors already in HBM.

value: algorithmic HBM GB/s sustained over the step
       (sum of iterations x B_pcg over both solves / step time;
       B_pcg = B_spmv + 11*8*n, B_spmv = nnz*12 + 4(n+1) + 16n).
layout: before timing, each input's SpMV layout is chosen by timing the
       plain store against 4..64 column panels (spk_csr_tune_layout; setup,
       reported with the candidates); --no-tune keeps the plain store.
roofline: the kernel pair that dominates the step -- the SpMV with the
       <p,q> epilogue and its one-block finisher, which every Jacobi-PCG
       step runs -- of the input whose pairs take the larger share of the
       step: B_spmv (algorithmic bytes, independent of the layout) / the
       time of one pair (all panel launches included) measured with HIP
       events on the library stream (the stream every kernel runs on); the
       plain SpMV's fraction is reported beside it.
sections (after the timed steps, not part of value): poisson_2d(256) PCG,
       mixed-precision GMRES(50)+ILU(0) on convection-diffusion 128^3,
       learned SPAI in FGMRES(30) on anisotropic diffusion 1024^2, batched
       PCG over 4096 systems.
cpu_baseline: the oracle's Jacobi-PCG (CPU restatement of the reference) on
       input (a) for a bounded number of iterations, one core.
"""
import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
# the network's output layer in the canonical parameter order
# W1[24][64] b1[64] W2[64][64] b2[64] W3[64][9] b3[9]
SPAI_W3 = 24 * 64 + 64 + 64 * 64 + 64
SPAI_B3 = SPAI_W3 + 64 * 9
# HBM-side bytes per call of the roofline kernel (the SpMV with the <p,q>
# epilogue) measured with rocprofv3 PMC counters (FETCH_SIZE x 2.0 +
# WRITE_SIZE, calibrated on a 256 MiB copy) at the layouts the tuner picks
# (plain CSR for the Poisson matrix, 16 column panels for the power-law
# one); the commands and the raw counts are in profiles/spmv_traffic_pmc.md
MEASURED_TRAFFIC = {"3D 7-point Poisson 192^3": 792.9e6,
                    "power-law SPD n=4194304": 12.39e9}
METRIC = ("time-to-1e-8 residual: learned-FGMRES vs Jacobi-PCG; "
          "SpMV GB/s % HBM peak")


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def b_spmv(n, nnz, s=8):
    return nnz * (s + 4) + 4 * (n + 1) + 2 * s * n


def b_pcg(n, nnz, s=8):
    return b_spmv(n, nnz, s) + 11 * s * n


CPU_LEGS = ("poisson192", "powerlaw", "aniso", "convdiff", "batched", "p2d")


def start_cpu_legs(legs):
    """Starts the oracle's CPU-baseline legs (oracle/cpu_baseline.py) as
    child processes before this process touches the GPU.  Each child pins
    itself to one host core (as taskset -c does) and runs its legs one
    after another; this process keeps the first two cores.  With fewer
    than three cores every leg runs in one child on the last core."""
    cores = sorted(os.sched_getaffinity(0))
    spare = cores[2:] or cores[-1:]
    groups = [legs[i::len(spare)] for i in range(min(len(spare), len(legs)))]
    procs = []
    for core, group in zip(spare, groups):
        cmd = [sys.executable, "-m", "oracle.cpu_baseline", ",".join(group),
               "--core", str(core)]
        procs.append((group, subprocess.Popen(
            cmd, cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE,
            text=True)))
    if len(cores) > 2:
        os.sched_setaffinity(0, set(cores[:2]))
    return {"procs": procs, "t0": time.perf_counter(), "nproc": len(cores),
            "cores": cores}


def collect_cpu_legs(state, deadline_s):
    """Waits for the legs (until deadline_s after they started); a leg
    still running then is stopped and reported unfinished."""
    out = {}
    for group, p in state["procs"]:
        so = se = None
        while so is None:  # a progress line every 30 s while a leg runs
            left = deadline_s - (time.perf_counter() - state["t0"])
            try:
                so, se = p.communicate(timeout=max(1.0, min(30.0, left)))
            except subprocess.TimeoutExpired:
                if left <= 30.0:
                    p.kill()
                    so, se = p.communicate()
                else:
                    log(f"cpu baseline: legs {','.join(group)} still running "
                        f"({time.perf_counter() - state['t0']:.0f} s)")
        for line in so.splitlines():
            try:
                r = json.loads(line)
                out[r["leg"]] = r
            except (ValueError, KeyError):
                pass
        for leg in group:
            if leg not in out:
                out[leg] = {"leg": leg, "unfinished": True,
                            "rc": p.returncode, "stderr": se[-300:]}
    return out


def attach_cpu_legs(out, legs):
    """GPU time beside the CPU leg of the same configuration."""
    def put(sec, leg, gpu_ms):
        r = legs.get(leg, {})
        if sec in out and isinstance(out[sec], dict) and r.get("s") and gpu_ms:
            out[sec]["cpu_" + leg] = {"s": r["s"],
                                      "extrapolated": bool(r.get("extrapolated")),
                                      "gpu_speedup": round(r["s"] * 1e3 / gpu_ms, 1)}
    p2 = out.get("poisson2d_pcg", {})
    put("poisson2d_pcg", "p2d", p2.get("ms"))
    mp = out.get("mixed_precision", {})
    put("mixed_precision", "convdiff",
        mp.get("fp64_gmres50_ilu0_mgs", {}).get("ms"))
    ls = out.get("learned_spai", {})
    put("learned_spai", "aniso", ls.get("jacobi_pcg_fp64", {}).get("ms"))
    bp = out.get("batched_pcg", {})
    put("batched_pcg", "batched", bp.get("fp64_graph", {}).get("ms"))


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(legs, state, inputs):
    """The headline's CPU figure: the oracle's Jacobi-PCG on input (a)
    (full solve) and input (b) (extrapolated from a sample), in the
    metric's unit, beside every leg's own report."""
    a, b = legs.get("poisson192", {}), legs.get("powerlaw", {})
    nproc = state["nproc"]
    res = {"unit": "GB/s", "cores": 1, "kind": "port",
           "cpu_model": cpu_model(), "nproc": nproc,
           "cores_note": f"1 of {nproc} cores per leg; legs ran at the same "
                         f"time, each pinned to its own core",
           "build": "oracle/liboracle.so, gcc -O3 -DNDEBUG -ffp-contract=off, "
                    "operator slots allocating and copying per call as the "
                    "reference's multiply / ilu_apply do",
           "legs": legs}
    if a.get("s") and b.get("s"):
        byt = 0.0
        for inp in inputs:
            leg = a if inp.name.startswith("3D") else b
            it = leg.get("iterations", POWERLAW_ITERS_CPU)
            byt += it * b_pcg(inp.n, inp.nnz)
        res["value"] = round(byt / (a["s"] + b["s"]) / 1e9, 3)
        res["sample"] = (f"Jacobi-PCG to 1e-8: (a) full solve, "
                         f"{a.get('iterations')} iterations in {a['s']:.1f} s; "
                         f"(b) extrapolated: {b.get('solver')} on a "
                         f"{b.get('sample_rows')}-row sample of the same law "
                         f"({b.get('sample_s')} s) scaled {b.get('scaling')} "
                         f"-> {b['s']:.1f} s")
        res["solve_s"] = round(a["s"] + b["s"], 3)
    elif a.get("s"):
        inp = [i for i in inputs if i.name.startswith("3D")][0]
        res["value"] = round(a["iterations"] * b_pcg(inp.n, inp.nnz) /
                             a["s"] / 1e9, 3)
        res["sample"] = (f"input (a) only: Jacobi-PCG full solve, "
                         f"{a['iterations']} iterations in {a['s']:.1f} s")
    else:
        res["value"] = None
        res["sample"] = "the CPU legs did not finish"
    return res


POWERLAW_ITERS_CPU = 11  # the power-law solve's Jacobi-PCG count


def layout_name(code):
    """'plain', 'panels:P' or 'tiles:SxW' for a layout code."""
    if code == 1:
        return "plain"
    if code > 1:
        return f"panels:{code}"
    return f"tiles:{-code // 65536}x{-code % 65536}"


class Input:
    def __init__(self, spk, name, A, tune=True, panels=None):
        self.name, self.A = name, A
        self.n, self.nnz = A.nrows, A.nnz
        self.layout = None
        if panels is not None:  # a fixed layout (profiling runs)
            A.set_layout(panels)
            self.layout = {"panels": panels, "fixed": True}
        elif tune:  # SpMV layout (column panels) chosen by timing, setup only
            t0 = time.perf_counter()
            chosen, tried = A.tune_layout()
            self.layout = {"panels": chosen, "name": layout_name(chosen),
                           "tried_us": {layout_name(p): round(us, 1)
                                        for p, us in tried},
                           "tune_s": round(time.perf_counter() - t0, 2)}
            log(f"{name}: SpMV layout {layout_name(chosen)} from {tried}")
        self.b = spk.uniform_pm1(42, self.n)
        self.x = spk.DeviceVector.zeros(self.n)
        self.J = spk.jacobi(A)
        self.cfg = spk.CGConfig(tolerance=1e-8, restart_iterations=20000,
                                max_iterations=20000)

    def solve(self, spk):
        spk._lib.call("spk_memset", self.x.ptr, 0, self.x.nbytes)
        return spk.conjugate_gradient(self.b, self.x, self.cfg, self.A,
                                      self.J, spk.identity)


def spmv_time(spk, A, x, reps):
    timer = spk.Timer()
    y = spk.DeviceVector(A.nrows)
    for _ in range(3):
        A.spmv(x, y)
    timer.start()
    for _ in range(reps):
        A.spmv(x, y)
    return timer.stop() / reps


def spmv_dot_time(spk, A, x, reps):
    """ms per fused q = A p, <p, q> launch pair (the SpMV with the dot in its
    epilogue and the one-block finisher that adds the block partials), the
    pair every Jacobi-PCG step of these inputs runs; HIP events on the
    library stream."""
    timer = spk.Timer()
    y = spk.DeviceVector(A.nrows)
    res = spk.DeviceVector(1)
    for _ in range(3):
        A.spmv_dot(x, y, res)
    timer.start()
    for _ in range(reps):
        A.spmv_dot(x, y, res)
    return timer.stop() / reps


def _mix(seed, k):
    """splitmix64 element k of the stream `seed` (the generators' RNG)."""
    m = (1 << 64) - 1
    z = (seed + (k + 1) * 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def speedup(res, base, other, target=1e-8):
    """base time / other time when both runs converged to the same FP64
    true-residual target; otherwise None, with the failed runs named."""
    a, b = res.get(base, {}), res.get(other, {})
    ok = [r.get("converged") and r.get("true_relres", 1.0) < target * 1.01
          for r in (a, b)]
    if all(ok):
        return round(a["ms"] / b["ms"], 3)
    failed = {k: {"converged": r.get("converged"),
                  "true_relres": r.get("true_relres")}
              for k, r, o in ((base, a, ok[0]), (other, b, ok[1])) if not o}
    res.setdefault("speedup_not_comparable", {})[f"{other}_vs_{base}"] = failed
    return None


def _timed(fn):
    t0 = time.perf_counter()
    r = fn()
    return r, (time.perf_counter() - t0) * 1e3


def ilu_schedules(spk, F, n, reps=3):
    """Times one FP64 and one FP32 application under each sweep schedule and
    keeps the faster for the solves."""
    timer = spk.Timer()
    out = {}
    for name in ("levels", "sync-free"):
        F.schedule = name
        for dt in (np.float64, np.float32):
            r = spk.DeviceVector.zeros(n, dt)
            z = spk.DeviceVector.zeros(n, dt)
            F.apply(r, z)
            timer.start()
            for _ in range(reps):
                F.apply(r, z)
            out[f"{name}_{np.dtype(dt).name}"] = round(timer.stop() / reps, 3)
    F.schedule = ("levels" if out["levels_float64"] <= out["sync-free_float64"]
                  else "sync-free")
    return out


def mixed_precision_section(spk, grid=128, seed=42):
    """Mixed-precision GMRES(50) + ILU(0) on 3D upwind convection-diffusion
    (grid^3, velocity (1, 0.5, 0.25), Peclet U[10,100] from the seed) to a
    1e-10 FP64 true residual: FP64 GMRES against FP32-inner / FP64-outer
    iterative refinement, and the refined solution's error against the FP64
    solve."""
    pe = 10.0 + 90.0 * ((_mix(seed ^ 0x5045, 0) >> 11) / 2.0 ** 53)
    h = 1.0 / (grid + 1)
    v = np.array([1.0, 0.5, 0.25])
    c = pe * h * v / np.linalg.norm(v)
    A = spk.convdiff_3d(grid, grid, grid, 1.0, *c)
    n = A.nrows
    b = spk.uniform_pm1(seed, n)
    F, t_ilu = _timed(lambda: spk.ilu0(A))
    sched = ilu_schedules(spk, F, n)
    log(f"ILU(0) {F.levels()} levels, apply ms per schedule {sched}, "
        f"using {F.schedule}")
    res = {"input": f"3D upwind convection-diffusion {grid}^3", "rows": n,
           "ilu0_levels": F.levels(), "ilu0_schedule": F.schedule,
           "ilu0_apply_ms": sched,
           "nnz": A.nnz, "peclet": round(pe, 3), "ilu0_setup_ms": round(t_ilu, 2),
           "target_true_relres": 1e-10}
    runs = [(0, "cgs2", spk.ORTHO_CGS2), (0, "mgs", spk.ORTHO_MGS)]
    runs += [(k, "cgs2", spk.ORTHO_CGS2) for k in (2, 3, 4)]
    # classical Gram-Schmidt once (half the passes over the basis): the
    # FP64 true residual of the refinement decides convergence
    runs += [(k, "cgs1", spk.ORTHO_CGS1) for k in (2, 3, 4)]
    timer = spk.Timer()
    for k, oname, ortho in runs:
        F.jacobi_sweeps = k
        tag = "ilu0" if k == 0 else f"ilu0jac{k}"
        if k:
            app = {}
            for dt in (np.float64, np.float32):
                r = spk.DeviceVector.zeros(n, dt)
                z = spk.DeviceVector.zeros(n, dt)
                F.apply(r, z)
                timer.start()
                for _ in range(3):
                    F.apply(r, z)
                app[np.dtype(dt).name] = round(timer.stop() / 3, 3)
            res[f"ilu0_jacobi{k}_apply_ms"] = app
        x64 = spk.DeviceVector.zeros(n)
        cfg = spk.GmresConfig(1e-10, 50, 5000, False, spk.F64, ortho)
        spk.gmres(b, spk.DeviceVector.zeros(n),
                  spk.GmresConfig(1e-10, 50, 50, False, spk.F64, ortho), A,
                  spk.identity, F)  # warm-up
        s64, t64 = _timed(lambda: spk.gmres(b, x64, cfg, A, spk.identity, F))
        r64 = spk.true_relres(A, b, x64)
        res[f"fp64_gmres50_{tag}_{oname}"] = {
            "iterations": s64.computed_iterations, "converged": s64.converged,
            "ms": round(t64, 2), "true_relres": r64}
        xir = spk.DeviceVector.zeros(n)
        icfg = spk.IrConfig(tolerance=1e-10, max_outer=20, inner_tolerance=1e-4,
                            restart=50, max_inner=2000,
                            inner_method=spk.IR_GMRES, orthogonalization=ortho)
        spk.ir_solve(b, spk.DeviceVector.zeros(n),
                     spk.IrConfig(1e-10, 1, 1e-2, 50, 50, spk.IR_GMRES, ortho),
                     A, F)
        sir, tir = _timed(lambda: spk.ir_solve(b, xir, icfg, A, F))
        rir = spk.true_relres(A, b, xir)
        a64, air = x64.numpy(), xir.numpy()
        res[f"ir_fp32_gmres50_{tag}_{oname}"] = {
            "outer_iterations": sir.outer_iterations,
            "inner_iterations": sir.inner_iterations,
            "converged": sir.converged, "ms": round(tir, 2), "true_relres": rir,
            "rel_error_vs_fp64_solve": float(np.linalg.norm(air - a64) /
                                             np.linalg.norm(a64))}
        res[f"speedup_ir_vs_fp64_{tag}_{oname}"] = speedup(
            res, f"fp64_gmres50_{tag}_{oname}", f"ir_fp32_gmres50_{tag}_{oname}",
            1e-10)
        log(f"mixed precision ({tag}, {oname}): FP64 GMRES "
            f"{s64.computed_iterations} it {t64:.1f} ms relres {r64:.2e}; IR "
            f"{sir.outer_iterations} outer {sir.inner_iterations} inner "
            f"{tir:.1f} ms relres {rir:.2e}")
    # the fastest form with the strict factors' values in FP16 for its FP32
    # passes (spk_ilu0_set_half_factors; the FP64 refinement is unchanged)
    F.jacobi_sweeps = 3
    F.half_factors = True
    xh = spk.DeviceVector.zeros(n)
    icfg = spk.IrConfig(tolerance=1e-10, max_outer=20, inner_tolerance=1e-4,
                        restart=50, max_inner=2000, inner_method=spk.IR_GMRES,
                        orthogonalization=spk.ORTHO_CGS2)
    spk.ir_solve(b, spk.DeviceVector.zeros(n),
                 spk.IrConfig(1e-10, 1, 1e-2, 50, 50, spk.IR_GMRES,
                              spk.ORTHO_CGS2), A, F)  # warm-up
    sh, th = _timed(lambda: spk.ir_solve(b, xh, icfg, A, F))
    res["ir_fp32_gmres50_ilu0jac3_fp16factors_cgs2"] = {
        "outer_iterations": sh.outer_iterations,
        "inner_iterations": sh.inner_iterations, "converged": sh.converged,
        "ms": round(th, 2), "true_relres": spk.true_relres(A, b, xh)}
    log(f"mixed precision (ilu0jac3, FP16 factors, cgs2): IR "
        f"{sh.outer_iterations} outer {sh.inner_iterations} inner {th:.1f} ms")
    F.half_factors = False
    F.jacobi_sweeps = 0
    # against the reference's method (FP64 GMRES(50), exact ILU(0) apply)
    base = min(res["fp64_gmres50_ilu0_cgs2"]["ms"],
               res["fp64_gmres50_ilu0_mgs"]["ms"])
    best = min((v["ms"], k) for k, v in res.items()
               if isinstance(v, dict) and v.get("converged")
               and v.get("true_relres", 1.0) < 1e-10 and "ms" in v)
    res["fastest_to_1e-10"] = {"solve": best[1], "ms": best[0],
                               "speedup_vs_fp64_exact_ilu0": round(base / best[0], 3)}
    return res


def learned_spai_section(spk, n_side=1024, train_side=256, train_count=512,
                         epochs=24, lr=2e-3, seed=4242, pcg_only=False):
    """Learned SPAI in FGMRES(30) on 2D anisotropic variable-coefficient
    diffusion (Q1, n_side^2 interior nodes, conductivity lognormal(0,1.5),
    anisotropy log-uniform [1,1e3], random rotation), trained on the device
    on train_count matrices of train_side^2 (seeds 0..train_count-1);
    compared with Jacobi-PCG, ILU(0)-PCG and FGMRES(30) with the untrained
    (Jacobi) network, each to a 1e-8 FP64 true residual; FGMRES
    orthogonalises by CGS2.  The guarded solve (spk_learned_solve) runs the
    same FGMRES behind the check of M and the stall monitor, and once with a
    poisoned network, whose M it rejects before falling back to Jacobi-PCG."""
    t0 = time.perf_counter()
    mats = [spk.aniso_q1_2d(train_side, s, 1.5) for s in range(train_count)]
    t_gen = time.perf_counter() - t0
    model = spk.SpaiModel(1)
    untrained = spk.SpaiModel(1)
    hist, t_train = _timed(lambda: model.train(mats, epochs=epochs,
                                               learning_rate=lr,
                                               shuffle_seed=7))
    spk.synchronize()
    # the same network trained on the loss of the operator PCG applies,
    # (1/n) ||I - S A||_F^2 with S = (M + M^T) / 2
    model_so = spk.SpaiModel(1)
    model_so.objective = spk.SPAI_LOSS_SYMMETRIC
    hist_so, t_train_so = _timed(lambda: model_so.train(
        mats, epochs=epochs, learning_rate=lr, shuffle_seed=7))
    spk.synchronize()
    del mats
    A = spk.aniso_q1_2d(n_side, seed, 1.5)
    n = A.nrows
    b = spk.uniform_pm1(42, n)
    Ml, t_pred = _timed(lambda: model.preconditioner(A))
    Mj = untrained.preconditioner(A)
    J = spk.jacobi(A)
    res = {"input": f"2D anisotropic Q1 diffusion {n_side}^2", "rows": n,
           "nnz": A.nnz, "train": {
               "matrices": train_count, "side": train_side, "epochs": epochs,
               "steps": len(hist), "learning_rate": lr,
               "generate_s": round(t_gen, 2), "train_s": round(t_train / 1e3, 3),
               "loss_first_epoch": float(np.mean(hist[:train_count])),
               "loss_last_epoch": float(np.mean(hist[-train_count:])),
               "symmetric_objective_train_s": round(t_train_so / 1e3, 3),
               "symmetric_objective_loss_last_epoch":
                   float(np.mean(hist_so[-train_count:]))},
           "predict_ms": round(t_pred, 2),
           "loss_test_learned": model.loss_grad(A)[0],
           "loss_test_jacobi": untrained.loss_grad(A)[0]}

    xref = {}

    def run(name, fn, warm=True):
        x = spk.DeviceVector.zeros(n)
        if warm:
            fn(x)  # warm-up (same solve)
            spk._lib.call("spk_memset", x.ptr, 0, x.nbytes)
        s, ms = _timed(lambda: fn(x))
        rel = spk.true_relres(A, b, x)
        xh = x.numpy()
        if not xref:  # the first run: FP64 Jacobi-PCG, the reference solve
            xref["x"] = xh
        err = float(np.linalg.norm(xh - xref["x"]) / np.linalg.norm(xref["x"]))
        it = getattr(s, "computed_iterations", None)
        d = {"ms": round(ms, 2), "true_relres": rel,
             "rel_error_vs_fp64_jacobi_pcg": err}
        if it is not None:
            d.update(iterations=it, converged=s.converged)
        else:
            d.update(outer=s.outer_iterations, inner=s.inner_iterations,
                     converged=s.converged)
        res[name] = d
        log(f"learned SPAI: {name}: {d}")

    cg = spk.CGConfig(1e-8, 50000, 50000)
    fg = spk.FgmresConfig(1e-8, 30, 50000, False, spk.F64, spk.ORTHO_CGS2)
    run("jacobi_pcg_fp64", lambda x: spk.conjugate_gradient(b, x, cg, A, J))
    # the learned inverse's symmetric part (SPD here) in the CG slot, FP64
    # and as FP32 PCG with FP64 reliable updates
    Msym, t_sym = _timed(lambda: model.predict(A).symmetric_part())
    Ms = spk.spai(Msym)
    res["symmetric_part_ms"] = round(t_sym, 2)
    run("learned_sym_pcg_fp64", lambda x: spk.conjugate_gradient(b, x, cg, A, Ms))
    rcfg = spk.IrConfig(tolerance=1e-8, max_outer=200, inner_tolerance=1e-2,
                        restart=0, max_inner=50000,
                        inner_method=spk.IR_CG_RELIABLE)
    run("jacobi_relcg_fp32", lambda x: spk.ir_solve(b, x, rcfg, A, J))
    run("learned_sym_relcg_fp32", lambda x: spk.ir_solve(b, x, rcfg, A, Ms))
    rcfg1 = spk.IrConfig(tolerance=1e-8, max_outer=200, inner_tolerance=1e-1,
                         restart=0, max_inner=50000,
                         inner_method=spk.IR_CG_RELIABLE)
    run("learned_sym_relcg_fp32_update_every_10x",
        lambda x: spk.ir_solve(b, x, rcfg1, A, Ms))
    # the same inverse with FP16 values in its FP32 SpMVs
    # (spk_csr_set_half_values): half of its value bytes per step
    Msym16 = model.predict(A).symmetric_part()
    Msym16.set_half_values(True)
    Ms16 = spk.spai(Msym16)
    run("learned_sym_relcg_fp32_update_every_10x_m_fp16",
        lambda x: spk.ir_solve(b, x, rcfg1, A, Ms16))
    # the network trained on the symmetric part's own loss
    Mso = spk.spai(model_so.predict(A).symmetric_part())
    run("learned_sym_pcg_fp64_symmetric_objective",
        lambda x: spk.conjugate_gradient(b, x, cg, A, Mso))
    Mso16_st = model_so.predict(A).symmetric_part()
    Mso16_st.set_half_values(True)
    Mso16 = spk.spai(Mso16_st)
    for k in ("learned_sym_pcg_fp64", "jacobi_relcg_fp32", "learned_sym_relcg_fp32",
              "learned_sym_relcg_fp32_update_every_10x",
              "learned_sym_relcg_fp32_update_every_10x_m_fp16"):
        res[f"speedup_{k}_vs_jacobi_pcg"] = speedup(res, "jacobi_pcg_fp64", k)
    if pcg_only:  # the PCG comparisons only (no ILU(0)-PCG, no FGMRES)
        return res
    F, t_ilu = _timed(lambda: spk.ilu0(A))
    res["ilu0_setup_ms"] = round(t_ilu, 2)
    res["ilu0_apply_ms"] = ilu_schedules(spk, F, n)
    res["ilu0_schedule"] = F.schedule
    res["ilu0_levels"] = F.levels()
    cgi = spk.CGConfig(1e-8, 200, 200)  # diverges: a bounded sample suffices
    run("ilu0_pcg_fp64", lambda x: spk.conjugate_gradient(b, x, cgi, A, F),
        warm=False)
    run("fgmres30_learned_fp64", lambda x: spk.fgmres(b, x, fg, A, Ml))
    # the untrained network (the Jacobi inverse) in the same slot: a bounded
    # sample (it does not converge on this matrix; 50,000 iterations left
    # it at 1.9e-5)
    fgu = spk.FgmresConfig(1e-8, 30, 3000, False, spk.F64, spk.ORTHO_CGS2)
    run("fgmres30_untrained_jacobi_fp64_3000_iterations",
        lambda x: spk.fgmres(b, x, fgu, A, Mj), warm=False)
    # the guarded solve: the same FGMRES behind the check of M and the stall
    # monitor (it needs no fallback here), and with a poisoned network (NaN
    # output layer), which falls back to Jacobi-PCG
    lcfg = spk.LearnedConfig(tolerance=1e-8, restart=30, max_iterations=50000)
    guard = {}

    def guarded(name, M, warm):
        def fn(x):
            guard[name] = spk.learned_solve(b, x, lcfg, A, M)
            return guard[name]
        run(name, fn, warm)
        g = guard[name]
        res[name].update(method=g.method, reasons=g.reasons,
                         learned_iterations=g.learned_iterations,
                         fallback_iterations=g.fallback_iterations,
                         converged=g.converged, true_relres=g.relres)

    # FGMRES's flexible slot holding a solve of its own: FP64 FGMRES(30) as
    # the refinement loop around FP32 PCG with the learned inverse's
    # symmetric part (up to k steps per application), against the same with
    # Jacobi inside
    inner = {}
    for k in (250, 500):
        for tag, Mi in (("learned", Ms), ("jacobi", J)):
            P = spk.inner_cg(A, Mi, iterations=k, precision=spk.F32)
            name = f"fgmres30_inner_pcg{k}_{tag}_fp32"
            run(name, lambda x: spk.fgmres(b, x, fg, A, P))
            inner[name] = P
            res[name]["inner_iterations_per_solve"] = \
                P.inner_iterations // 2  # warm-up + timed solve
    # the flexible slot holding FP32 PCG with FP64 reliable updates and the
    # learned inverse's symmetric part (spk_precond_create_inner_ir), each
    # application to a relative tolerance: 1e-4 (FGMRES takes a few outer
    # steps) or 1e-8 (one outer step; FGMRES checks the true residual)
    for tol in (1e-4, 1e-8):
        icfg = spk.IrConfig(tolerance=tol, max_outer=200, inner_tolerance=1e-1,
                            restart=0, max_inner=50000,
                            inner_method=spk.IR_CG_RELIABLE)
        for tag, Mi in (("learned", Ms), ("learned_m_fp16", Ms16),
                        ("learned_symmetric_objective_m_fp16", Mso16)):
            P = spk.inner_ir(A, Mi, icfg)
            name = f"fgmres30_inner_relcg_to_{tol:g}_{tag}_fp32"
            run(name, lambda x: spk.fgmres(b, x, fg, A, P))
            inner[name] = P
            res[name]["inner_iterations_per_solve"] = P.inner_iterations // 2
    guarded("guarded_fgmres30_learned", Ml, False)  # FGMRES above: warm
    poisoned = spk.SpaiModel(1)
    pp = model.params
    pp[SPAI_W3:SPAI_B3] = np.nan
    poisoned.params = pp
    guarded("guarded_fgmres30_nan_network", poisoned.preconditioner(A), True)
    # the metric's own ratio: learned-SPAI FGMRES against Jacobi-PCG, both
    # to the 1e-8 FP64 true residual
    res["plain_learned_fgmres_vs_jacobi_pcg"] = speedup(
        res, "jacobi_pcg_fp64", "fgmres30_learned_fp64")
    best = min((res[k]["ms"], k) for k in
               ["fgmres30_learned_fp64"] + [k for k in inner if "learned" in k]
               if res[k].get("converged") and res[k]["true_relres"] < 1.01e-8)
    res["learned_fgmres_vs_jacobi_pcg"] = {
        "solve": best[1], "ratio": speedup(res, "jacobi_pcg_fp64", best[1]),
        "outer_iterations": res[best[1]]["iterations"], "target": 2.0}
    # the same among the forms where FGMRES itself takes two or more steps
    multi = min((res[k]["ms"], k) for k in
                ["fgmres30_learned_fp64"] + [k for k in inner if "learned" in k]
                if res[k].get("converged") and res[k]["true_relres"] < 1.01e-8
                and res[k]["iterations"] >= 2)
    res["learned_fgmres_vs_jacobi_pcg_two_or_more_outer"] = {
        "solve": multi[1], "ratio": speedup(res, "jacobi_pcg_fp64", multi[1]),
        "outer_iterations": res[multi[1]]["iterations"]}
    res["fallback_overhead_vs_jacobi_pcg"] = speedup(
        res, "jacobi_pcg_fp64", "guarded_fgmres30_nan_network")
    return res


def short_index_section(spk, reps=50):
    """SpMV time with 16-bit column offsets (spk_csr_set_short_indices)
    against the 32-bit indices, FP64 and FP32, on banded natural-order
    stencil matrices (mean of reps calls after 5 warm-up calls; the results
    are equal bit for bit)."""
    def t(A, dt):
        x = spk.DeviceVector.from_numpy(np.ones(A.ncols, dt))
        y = spk.DeviceVector.zeros(A.nrows, dt)
        for _ in range(5):
            A.spmv(x, y)
        spk.synchronize()
        t0 = time.perf_counter()
        for _ in range(reps):
            A.spmv(x, y)
        spk.synchronize()
        return (time.perf_counter() - t0) / reps * 1e6
    res = {}
    for name, mk in (
            ("2D anisotropic Q1 2048^2", lambda: spk.aniso_q1_2d(2048, 7, 1.5)),
            ("3D 7-point Poisson 160^3", lambda: spk.poisson_3d(160, 160, 160)),
            ("2D anisotropic Q1 1024^2", lambda: spk.aniso_q1_2d(1024, 4242, 1.5)),
            ("3D upwind convection-diffusion 128^3",
             lambda: spk.convdiff_3d(128, 128, 128, 1.0, 0.3, 0.15, 0.07))):
        A = mk()
        d = {"rows": A.nrows, "nnz": A.nnz}
        for dt in (np.float64, np.float32):
            a = t(A, dt)
            A.set_short_indices(True)
            b = t(A, dt)
            A.set_short_indices(False)
            k = np.dtype(dt).name
            d[k] = {"int32_us": round(a, 1), "short_us": round(b, 1),
                    "speedup": round(a / b, 3)}
        res[name] = d
        log(f"short indices: {name}: {d}")
        del A
    return res


def krylov_section(spk, grid=128, seed=7):
    """The other Krylov solvers on the device, FP64 + Jacobi to a 1e-8
    relative residual: nonsymmetric 3D upwind convection-diffusion grid^3
    (Peclet as the mixed-precision section) with BiCGSTAB, CGS, BiCG and
    QMR; the SPD 3D Poisson grid^3 with CG and MINRES.  Times are whole
    solves (warm), counts are the solvers' own (matvecs for the two-sided
    methods)."""
    pe = 10.0 + 90.0 * ((_mix(42 ^ 0x5045, 0) >> 11) / 2.0 ** 53)
    h = 1.0 / (grid + 1)
    v = np.array([1.0, 0.5, 0.25])
    c = pe * h * v / np.linalg.norm(v)
    res = {}
    for name, A in ((f"3D upwind convection-diffusion {grid}^3",
                     spk.convdiff_3d(grid, grid, grid, 1.0, *c)),
                    (f"3D 7-point Poisson {grid}^3", spk.poisson_3d(grid, grid, grid))):
        n = A.nrows
        b = spk.uniform_pm1(seed, n)
        J = spk.jacobi(A)
        At = A.transpose()
        cfg = spk.BicgstabConfig(1e-8, 20000)
        if name.startswith("3D upwind"):
            runs = (("bicgstab", lambda x: spk.bicgstab(b, x, cfg, A, J)),
                    ("cgs", lambda x: spk.cgs(b, x, cfg, A, J)),
                    ("bicg", lambda x: spk.bicg(b, x, cfg, A, At, J)),
                    ("qmr", lambda x: spk.qmr(b, x, cfg, A, At, J)))
        else:
            cgc = spk.CGConfig(1e-8, 20000, 20000)
            runs = (("cg", lambda x: spk.conjugate_gradient(b, x, cgc, A, J)),
                    ("minres", lambda x: spk.minres(b, x, cfg, A, J)))
        out = {"rows": n, "nnz": A.nnz}
        for sname, fn in runs:
            x = spk.DeviceVector.zeros(n)
            fn(x)
            spk._lib.call("spk_memset", x.ptr, 0, x.nbytes)
            s, ms = _timed(lambda: fn(x))
            rel = spk.true_relres(A, b, x)
            out[sname] = {"ms": round(ms, 2), "iterations": s.computed_iterations,
                          "converged": s.converged, "true_relres": rel,
                          "breakdown": s.breakdown}
            log(f"krylov: {name}: {sname} {s.computed_iterations} it "
                f"{ms:.1f} ms relres {rel:.2e}")
        res[name] = out
    return res


def mmio_section(spk, grid=96):
    """Matrix Market text through a device store: write the 3D Poisson
    grid^3 store as text, read it back (host scan + device assembly), and
    check the pattern and values round-trip."""
    A = spk.poisson_3d(grid, grid, grid)
    t, t_w = _timed(lambda: A.to_matrix_market_text())
    B, t_r = _timed(lambda: spk.CsrMatrix.from_matrix_market_text(t))
    ra, ca, va = A.download()
    rb, cb, vb = B.download()
    same = bool(np.array_equal(ra, rb) and np.array_equal(ca, cb)
                and np.array_equal(va, vb))
    mb = len(t) / 1e6
    log(f"matrix market: {A.nnz} entries, {mb:.0f} MB text, write "
        f"{t_w:.0f} ms, read {t_r:.0f} ms, round trip exact: {same}")
    return {"input": f"3D 7-point Poisson {grid}^3", "entries": A.nnz,
            "text_MB": round(mb, 1), "write_ms": round(t_w, 1),
            "read_ms": round(t_r, 1), "read_MB_s": round(mb / (t_r / 1e3), 1),
            "round_trip_exact": same}


def frobenius_optimal_spai(n, rp, ci, v):
    """The SPAI the network's loss aims at, computed exactly: row i of M
    minimises ||e_i^T - m_i^T A||_2 over the pattern J of row i of A, i.e.
    (A A^T)[J, J] m = A[J, i] -- one small SPD system per row, solved in
    batches (rows padded to the widest with identity rows)."""
    import scipy.sparse as sps
    A = sps.csr_matrix((v, ci, rp), shape=(n, n))
    B = (A @ A.T).tocsr()
    lens = np.diff(rp)
    W = int(lens.max())
    J = -np.ones((n, W), np.int64)
    pos = np.arange(len(ci)) - np.repeat(rp[:-1], lens)
    J[np.repeat(np.arange(n), lens), pos] = ci
    ok = J >= 0
    Jc = np.where(ok, J, 0)
    G = np.zeros((n, W, W))
    for a in range(W):
        for c in range(W):
            g = np.asarray(B[Jc[:, a], Jc[:, c]]).ravel()
            G[:, a, c] = np.where(ok[:, a] & ok[:, c], g, 0.0)
        G[:, a, a] = np.where(ok[:, a], G[:, a, a], 1.0)
    rhs = np.asarray(A[Jc.ravel(), np.repeat(np.arange(n), W)]).reshape(n, W)
    m = np.linalg.solve(G, np.where(ok, rhs, 0.0)[:, :, None])[:, :, 0]
    return m[ok]


def spai_ceiling_section(spk, n_side=1024, train_side=256, train_count=512,
                         epochs=24, lr=2e-3, seed=4242):
    """How close the learned SPAI is to the best SPAI on A's pattern: the
    loss (1/n)||I - M A||_F^2 of Jacobi, of the trained network and of the
    Frobenius-optimal M (computed exactly on the host), and FP64 PCG to
    1e-8 with the symmetric part of each."""
    import scipy.sparse as sps
    A = spk.aniso_q1_2d(n_side, seed, 1.5)
    n = A.nrows
    rp, ci, v = A.download()
    rp, ci = rp.astype(np.int64), ci.astype(np.int64)
    mv, t_exact = _timed(lambda: frobenius_optimal_spai(n, rp, ci, v))
    mats = [spk.aniso_q1_2d(train_side, s, 1.5) for s in range(train_count)]
    model = spk.SpaiModel(1)
    model.train(mats, epochs=epochs, learning_rate=lr, shuffle_seed=7)
    spk.synchronize()
    del mats
    Ml = model.predict(A)
    diag = np.repeat(np.arange(n), np.diff(rp)) == ci
    jac = np.zeros_like(v)
    jac[diag] = 1.0 / v[diag]
    Ad = sps.csr_matrix((v, ci, rp), shape=(n, n))

    def loss(m):
        R = sps.identity(n, format="csr") - sps.csr_matrix((m, ci, rp), shape=(n, n)) @ Ad
        return round(float(R.multiply(R).sum() / n), 4)

    res = {"input": f"2D anisotropic Q1 diffusion {n_side}^2", "rows": n,
           "exact_spai_host_s": round(t_exact / 1e3, 1),
           "loss": {"jacobi": loss(jac), "learned": loss(Ml.download()[2]),
                    "frobenius_optimal": loss(mv)}}
    Me = spk.CsrMatrix.from_host(n, n, rp.astype(np.int32), ci.astype(np.int32), mv)
    b = spk.uniform_pm1(42, n)
    cg = spk.CGConfig(1e-8, 50000, 50000)
    for name, M in (("jacobi", spk.jacobi(A)),
                    ("learned_sym", spk.spai(Ml.symmetric_part())),
                    ("frobenius_optimal_sym", spk.spai(Me.symmetric_part()))):
        x = spk.DeviceVector.zeros(n)
        s, ms = _timed(lambda: spk.conjugate_gradient(b, x, cg, A, M))
        res["pcg_" + name] = {"iterations": s.computed_iterations,
                              "converged": bool(s.converged), "ms": round(ms, 1),
                              "true_relres": spk.true_relres(A, b, x)}
        log(f"SPAI ceiling: PCG {name}: {res['pcg_' + name]}")
    log(f"SPAI ceiling: loss {res['loss']}")
    return res


def rcm_section(spk, grid=128, seed=5):
    """Reverse Cuthill-McKee on the device: the 3D Poisson grid^3 under a
    seeded random relabelling (a scrambled band), reordered by RCM and
    permuted back with dperm; bandwidth before and after."""
    A0 = spk.poisson_3d(grid, grid, grid)
    n = A0.nrows
    lab = np.random.default_rng(seed).permutation(n)
    A = A0.permute(lab, "both")

    def band(M):
        rp, ci, _ = M.download()
        rows = np.repeat(np.arange(M.nrows), np.diff(rp))
        return int(np.abs(ci - rows).max())

    perm, t_rcm = _timed(lambda: A.rcm())
    B, t_perm = _timed(lambda: A.permute(perm, "both"))
    out = {"input": f"3D 7-point Poisson {grid}^3, randomly relabelled",
           "rows": n, "nnz": A.nnz, "rcm_ms": round(t_rcm, 1),
           "dperm_ms": round(t_perm, 1), "bandwidth_scrambled": band(A),
           "bandwidth_rcm": band(B), "bandwidth_natural": band(A0)}
    log(f"rcm: {n} rows in {t_rcm:.0f} ms, bandwidth {out['bandwidth_scrambled']}"
        f" -> {out['bandwidth_rcm']} (natural {out['bandwidth_natural']})")
    return out


def poisson2d_rhs(spk, n, seed=42):
    """splitmix64 uniform[-1,1] minus its mean: orthogonal to the constant
    null vector of the Neumann poisson_2d (matgen.hpp:211)."""
    b = spk.uniform_pm1(seed, n).numpy()
    return spk.DeviceVector.from_numpy(b - b.mean())


def poisson2d_section(spk, side=256):
    """Jacobi-PCG on poisson_2d(side) (the reference's own CPU-runnable
    case), to 1e-8 with restart_iterations = max_iterations = 20000."""
    A = spk.poisson_2d(side)
    b = poisson2d_rhs(spk, A.nrows)
    J = spk.jacobi(A)
    cfg = spk.CGConfig(1e-8, 20000, 20000)
    x = spk.DeviceVector.zeros(A.nrows)
    spk.conjugate_gradient(b, x, cfg, A, J)
    spk._lib.call("spk_memset", x.ptr, 0, x.nbytes)
    s, ms = _timed(lambda: spk.conjugate_gradient(b, x, cfg, A, J))
    res = {"input": f"poisson_2d({side}) (Neumann), mean-free RHS",
           "rows": A.nrows, "nnz": A.nnz, "iterations": s.computed_iterations,
           "converged": s.converged, "ms": round(ms, 2),
           "true_relres": spk.true_relres(A, b, x)}
    log(f"poisson_2d({side}): {s.computed_iterations} it {ms:.1f} ms")
    return res


def batched_section(spk, count=4096, seed=42, smin=32, smax=256,
                    sample=256, reps=3):
    """Batched Jacobi-PCG over `count` 2D variable-coefficient diffusion
    systems (sides U{smin..smax}, lognormal(0,1) conductivity, Dirichlet) in
    one persistent hipGraph-replayed launch: FP32 SpMV/vectors with FP64
    reliable updates (true residual, x accumulation), 1e-8 FP64 true residual
    per system; launch shape from the autotuner.  Compared with the same
    kernel in FP64 throughout."""
    (B, t_gen) = _timed(lambda: spk.BatchedSystems.diffusion(count, seed,
                                                             smin, smax))
    n, nnz = B.total_rows, B.nnz
    b = spk.uniform_pm1(seed, n)
    x = spk.DeviceVector.zeros(n)
    cfg = spk.BatchConfig(1e-8, 1e-2, 30, 20000, spk.F32)
    (tune, t_tune) = _timed(lambda: B.autotune(cfg, b, x, sample=sample))
    chosen, tried = tune
    res = {"input": f"{count} systems, 2D 5-point variable-coefficient "
                    f"diffusion, sides U{{{smin}..{smax}}}",
           "systems": count, "rows": n, "nnz": nnz,
           "generate_ms": round(t_gen, 1), "autotune_ms": round(t_tune, 1),
           "tuning": {"block": chosen[0], "wg_per_cu": chosen[1],
                      "lds_rows": chosen[2]},
           "tuning_candidates": len(tried)}
    timer = spk.Timer()

    def run(c, graph):
        B.solve(c, b, x, use_graph=graph, summary=False)  # capture / warm-up
        ms = []
        for _ in range(reps):
            timer.start()
            B.solve(c, b, x, use_graph=graph, summary=False)
            ms.append(timer.stop())
        s = B.solve(c, b, x, use_graph=graph)
        return float(np.median(ms)), s

    # residual reduction of the FP32 recurrence between two FP64 true-residual
    # updates (reliable updates; the search direction is kept)
    tries = {}
    for itol in (1e-2, 1e-4):
        c = spk.BatchConfig(1e-8, itol, 30, 20000, spk.F32)
        tries[itol] = run(c, True)
        log(f"batched FP32-inner, reduction between FP64 updates {itol:g}: "
            f"{tries[itol][0]:.1f} ms, {tries[itol][1]['total_inner_iterations']}"
            f" it, {tries[itol][1]['total_outer_iterations']} outer")
    best = min(tries, key=lambda k: tries[k][0])
    res["fp32_inner_by_update_reduction_ms"] = {f"{k:g}": round(v[0], 2)
                                               for k, v in tries.items()}
    res["inner_tolerance"] = best
    cfg = spk.BatchConfig(1e-8, best, 30, 20000, spk.F32)
    ms32, s32 = run(cfg, True)
    # bytes per inner iteration of a system with n_k rows, nnz_k entries:
    # FP32 SpMV (nnz*(4+4) + 4(n+1)) + 11 vector words of 4 bytes
    it, ou, rr, cv = B.results()
    x32 = x.numpy()
    ro = B.row_offsets()
    rows_k = np.diff(ro)
    nnz_k = 5 * rows_k - 4 * np.sqrt(rows_k)
    bytes_it = nnz_k * 8 + 4 * (rows_k + 1) + 44 * rows_k
    tot = float(np.sum(it * bytes_it))
    gbs = tot / (ms32 * 1e-3) / 1e9
    # what the kernel moves through HBM per inner iteration and row: the
    # sliced-ELL matrix (5 slots x (4-byte value + 2-byte column offset):
    # every column of these grids lies within 256 of its row), q written,
    # the d/r pass
    # (d, r, q, 1/diag read, d, r written) and the p pass (r, 1/diag read);
    # p itself (read by the gathers and both passes, written by the p pass)
    # stays in LDS for systems up to lds_rows rows, else adds 16 bytes
    lds_rows = chosen[2]
    per_row = 5 * 6 + 4 + 24 + 8 + np.where(rows_k <= lds_rows, 0, 16)
    tot_hbm = float(np.sum(it * rows_k * per_row))
    gbs_hbm = tot_hbm / (ms32 * 1e-3) / 1e9
    res["fp32_inner_graph"] = {
        "ms": round(ms32, 2), "converged": s32["converged"],
        "max_true_relres": s32["max_relres"],
        "inner_iterations": s32["total_inner_iterations"],
        "max_inner_iterations": s32["max_inner_iterations"],
        "outer_iterations": s32["total_outer_iterations"],
        "algorithmic_GBs": round(gbs, 1),
        "frac_hbm_peak": round(gbs / HBM_PEAK_GBS, 4),
        "hbm_model_GBs": round(gbs_hbm, 1),
        "hbm_model_frac_peak": round(gbs_hbm / HBM_PEAK_GBS, 4),
        "hbm_model": "per inner iteration and row: 30 B sliced-ELL matrix "
                     "(FP32 values, 16-bit column offsets) + "
                     "4 B q + 24 B d/r pass + 8 B p pass, +16 B of p for "
                     f"systems above {lds_rows} rows (p in LDS below)"}
    c64 = spk.BatchConfig(1e-8, 1e-8, 3, 20000, spk.F64)
    ms64, s64 = run(c64, True)
    res["fp64_graph"] = {"ms": round(ms64, 2), "converged": s64["converged"],
                         "max_true_relres": s64["max_relres"],
                         "inner_iterations": s64["total_inner_iterations"]}
    # the FP32-inner solution against the FP64 solve, per system
    x64 = x.numpy()
    d2 = np.add.reduceat((x32 - x64) ** 2, ro[:-1])
    n2 = np.add.reduceat(x64 ** 2, ro[:-1])
    rel = np.sqrt(d2 / np.maximum(n2, 1e-300))
    res["fp32_vs_fp64_solution"] = {
        "max_rel_error": float(rel.max()), "median_rel_error": float(np.median(rel)),
        "note": "per system ||x32 - x64|| / ||x64||, both solved to a 1e-8 "
                "FP64 true residual"}
    both = s32["converged"] == count and s64["converged"] == count
    res["speedup_fp32_inner_vs_fp64"] = round(ms64 / ms32, 3) if both else None
    log(f"batched: {count} systems n={n} nnz={nnz}: tuned {chosen} "
        f"({t_tune:.0f} ms); FP32-inner {ms32:.1f} ms "
        f"{s32['total_inner_iterations']} it ({gbs:.0f} GB/s), FP64 "
        f"{ms64:.1f} ms, max relres {s32['max_relres']:.2e}")
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--grid", type=int, default=192)
    ap.add_argument("--powerlaw-n", type=int, default=4194304)
    ap.add_argument("--inputs", default="ab", help="a, b or ab")
    ap.add_argument("--spmv-reps", type=int, default=30)
    ap.add_argument("--no-cpu", action="store_true",
                    help="skip the CPU baseline legs")
    ap.add_argument("--cpu-legs", default=",".join(CPU_LEGS),
                    help="oracle legs timed on host cores beside the GPU "
                         "work: " + ",".join(CPU_LEGS))
    ap.add_argument("--cpu-deadline", type=float, default=480.0,
                    help="seconds after start when unfinished legs stop")
    ap.add_argument("--no-tune", action="store_true",
                    help="keep the plain CSR layout (no column panels)")
    ap.add_argument("--panels", default=None,
                    help="fixed SpMV layouts instead of the tuner's choice, "
                         "one per input: e.g. 1,16 (profiling runs); a "
                         "negative code -(slots * 65536 + window) selects "
                         "window tiles")
    ap.add_argument("--sections",
                    default="p2d,mp,spai,batched,krylov,mmio,rcm,short-idx",
                    help="extra measurements after the timed steps: "
                         "p2d (poisson_2d(256) PCG), mp (mixed precision), "
                         "spai (learned SPAI), spai-pcg (its PCG "
                         "comparisons only), "
                         "batched (batched PCG), krylov (BiCGSTAB, CGS, "
                         "BiCG, QMR, CG, MINRES), mmio (Matrix Market "
                         "round trip), rcm (device reverse Cuthill-McKee), "
                         "short-idx (SpMV with 16-bit column offsets), "
                         "spai-ceiling (learned vs Frobenius-optimal SPAI; "
                         "not in the default list); 'none' for neither")
    ap.add_argument("--spai-epochs", type=int, default=24)
    ap.add_argument("--spai-train", type=int, default=512)
    ap.add_argument("--spai-side", type=int, default=1024)
    ap.add_argument("--mp-grid", type=int, default=128)
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path "
              "(every run uses exactly one MI355X); use --gpus 1",
              file=sys.stderr)
        sys.exit(2)

    # the CPU legs start first, in child processes pinned to their own
    # cores, and run while the GPU is measured
    legs_state = None
    if not args.no_cpu:
        legs_state = start_cpu_legs([g for g in args.cpu_legs.split(",") if g])
    import sparkit_amd as spk
    spk.init(0)
    cus, name = spk.device_info()
    log(f"device: {name}, {cus} CUs")
    inputs = []
    # one fixed layout per selected input, in the order a, b
    fixed_panels = ([int(p) for p in args.panels.split(",")]
                    if args.panels else []) + [None, None]
    if "a" in args.inputs:
        t0 = time.perf_counter()
        A = spk.poisson_3d(args.grid)
        log(f"(a) poisson_3d({args.grid}): n={A.nrows} nnz={A.nnz} "
            f"built in {time.perf_counter() - t0:.2f} s")
        inputs.append(Input(spk, f"3D 7-point Poisson {args.grid}^3", A,
                            not args.no_tune, fixed_panels.pop(0)))
    if "b" in args.inputs:
        t0 = time.perf_counter()
        A = spk.powerlaw_spd(args.powerlaw_n, 42)
        nb, nl = A.plan_info()
        log(f"(b) powerlaw_spd({args.powerlaw_n}): n={A.nrows} nnz={A.nnz} "
            f"({A.nnz / A.nrows:.1f}/row, {nl} long rows) built in "
            f"{time.perf_counter() - t0:.2f} s")
        inputs.append(Input(spk, f"power-law SPD n={args.powerlaw_n}", A,
                            not args.no_tune, fixed_panels.pop(0)))

    timer = spk.Timer()
    for _ in range(args.warmup):
        for inp in inputs:
            inp.solve(spk)
    spk.synchronize()
    step_ms, per = [], {inp.name: {"ms": [], "it": []} for inp in inputs}
    t_all0 = time.perf_counter()
    for k in range(args.steps):
        timer.start()
        for inp in inputs:
            t0 = time.perf_counter()
            s = inp.solve(spk)
            per[inp.name]["ms"].append((time.perf_counter() - t0) * 1e3)
            per[inp.name]["it"].append(s.computed_iterations)
            assert s.converged, f"{inp.name} did not converge"
        ms = timer.stop()
        step_ms.append(ms)
        log(f"step {k}: {ms:.2f} ms " + ", ".join(
            f"{nm}: {v['it'][-1]} it {v['ms'][-1]:.1f} ms"
            for nm, v in per.items()))
    spk.synchronize()
    wall = time.perf_counter() - t_all0
    ms_step = float(np.mean(step_ms))
    total_bytes = sum(np.mean(per[inp.name]["it"]) * b_pcg(inp.n, inp.nnz)
                      for inp in inputs)
    value = total_bytes / (ms_step * 1e-3) / 1e9

    results, dom, dom_share = [], None, -1.0
    for inp in inputs:
        us = spmv_time(spk, inp.A, inp.x, args.spmv_reps) * 1e3
        dus = spmv_dot_time(spk, inp.A, inp.x, args.spmv_reps) * 1e3
        bs = b_spmv(inp.n, inp.nnz)
        gbs = bs / (us * 1e-6) / 1e9
        dgbs = bs / (dus * 1e-6) / 1e9
        relres = spk.true_relres(inp.A, inp.b, inp.x)
        it = int(np.median(per[inp.name]["it"]))
        share = it * dus * 1e-3 / ms_step
        r = {"input": inp.name, "rows": inp.n, "nnz": inp.nnz,
             "pcg_iterations": it,
             "pcg_time_to_1e-8_ms": round(float(np.mean(per[inp.name]["ms"])), 3),
             "true_relres": relres,
             "spmv_us": round(us, 2), "spmv_GBs": round(gbs, 1),
             "spmv_frac_hbm_peak": round(gbs / HBM_PEAK_GBS, 4),
             "spmv_dot_us": round(dus, 2), "spmv_dot_GBs": round(dgbs, 1),
             "spmv_dot_frac_hbm_peak": round(dgbs / HBM_PEAK_GBS, 4),
             "spmv_bytes": bs, "spmv_layout": inp.layout}
        if gbs > HBM_PEAK_GBS:
            r["spmv_rate_note"] = ("the CSR form's bytes over the time; a store "
                                   "whose rows repeat reads one byte a row")
        panels = inp.A.panels
        if panels > 1:
            # rows scatter over all columns: every product is a random
            # gather, bounded by the gather rate at the layout's x window
            w = -(-inp.A.ncols // panels)
            gps, _ = spk.gather_rate(w)
            gps_full, _ = spk.gather_rate(inp.A.ncols)
            ach = inp.nnz / (us * 1e-6)
            r["gather_ceiling"] = {
                "window_doubles": w, "ceiling_Ggathers_s": round(gps / 1e9, 2),
                "ceiling_full_x_Ggathers_s": round(gps_full / 1e9, 2),
                "spmv_Ggathers_s": round(ach / 1e9, 2),
                "frac": round(ach / gps, 4)}
            log(f"{inp.name}: {ach / 1e9:.1f} G gathers/s against a "
                f"{gps / 1e9:.1f} G/s ceiling at a {w}-entry window "
                f"({gps_full / 1e9:.1f} G/s over all of x)")
        results.append(r)
        log(f"{inp.name}: spmv {us:.1f} us {gbs:.0f} GB/s "
            f"({gbs / HBM_PEAK_GBS:.1%}), relres {relres:.2e}")
        if share > dom_share:
            dom, dom_share = r, share

    # device-to-device copy (the runtime's blit kernel): practical ceiling
    cbytes = 256 * 1024 * 1024
    ca, cb = spk.DeviceVector(cbytes // 8), spk.DeviceVector(cbytes // 8)
    spk._lib.call("spk_memset", ca.ptr, 0, cbytes)
    for _ in range(3):
        spk._lib.call("spk_memcpy_dtod", cb.ptr, ca.ptr, cbytes)
    timer.start()
    for _ in range(20):
        spk._lib.call("spk_memcpy_dtod", cb.ptr, ca.ptr, cbytes)
    copy_gbs = 2 * cbytes / (timer.stop() / 20 * 1e-3) / 1e9
    log(f"copy: {copy_gbs:.0f} GB/s (read+write)")

    out = {
        "metric": METRIC,
        "value": round(float(value), 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_step, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (device-generated matrices, splitmix64 RHS)",
        "config": {"workload": "FP64 CSR SpMV + Jacobi-PCG to 1e-8 on " +
                               " and ".join(i.name for i in inputs),
                   "index": "int32", "inputs": results,
                   "parallelism": "1 GPU"},
        "roofline": {"bound": "hbm",
                     "kernel": "spmv_kernel with the <p,q> epilogue + its "
                               f"one-block finisher ({dom['input']}; the pair "
                               "each PCG step runs)",
                     "achieved": dom["spmv_dot_GBs"], "peak": HBM_PEAK_GBS,
                     "unit": "GB/s",
                     "frac": round(dom["spmv_dot_GBs"] / HBM_PEAK_GBS, 4),
                     "algorithmic_bytes": dom["spmv_bytes"],
                     "launch_us": dom["spmv_dot_us"],
                     "plain_spmv_frac": dom["spmv_frac_hbm_peak"],
                     "traffic": MEASURED_TRAFFIC.get(dom["input"]),
                     "traffic_source": "profiles/spmv_traffic_pmc.md"
                     if dom["input"] in MEASURED_TRAFFIC else None},
        "copy_GBs": round(copy_gbs, 1),
        "wall_s_timed": round(wall, 3),
    }
    secs = args.sections.split(",")

    def section(key, fn):
        # a failing section is reported in the line, not fatal to it
        try:
            out[key] = fn()
        except Exception as e:  # noqa: BLE001
            log(f"section {key} failed: {e}")
            out[key] = {"error": str(e)}

    if "p2d" in secs:
        section("poisson2d_pcg", lambda: poisson2d_section(spk))
    if "mp" in secs:
        section("mixed_precision",
                lambda: mixed_precision_section(spk, args.mp_grid))
    if "spai" in secs or "spai-pcg" in secs:
        section("learned_spai", lambda: learned_spai_section(
            spk, n_side=args.spai_side, train_count=args.spai_train,
            epochs=args.spai_epochs, pcg_only="spai" not in secs))
    if "batched" in secs:
        section("batched_pcg", lambda: batched_section(spk))
    if "krylov" in secs:
        section("krylov_solvers", lambda: krylov_section(spk))
    if "mmio" in secs:
        section("matrix_market", lambda: mmio_section(spk))
    if "rcm" in secs:
        section("rcm", lambda: rcm_section(spk))
    if "short-idx" in secs:
        section("short_indices", lambda: short_index_section(spk))
    if "spai-ceiling" in secs:
        section("spai_ceiling", lambda: spai_ceiling_section(
            spk, n_side=args.spai_side, train_count=args.spai_train,
            epochs=args.spai_epochs))
    if legs_state is not None:
        log("cpu baseline: waiting for the legs ...")
        legs = collect_cpu_legs(legs_state, args.cpu_deadline)
        out["cpu_baseline"] = cpu_baseline(legs, legs_state, inputs)
        attach_cpu_legs(out, legs)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
