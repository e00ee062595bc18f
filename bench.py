#!/usr/bin/env python3
"""Throughput of the per-time-step hot path on one MI355X, FP64 and mixed precision.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--cfg 2] [--no-cpu]

A step is one RK2 time step (two projection stages: Smagorinsky eddy
viscosity, advection/diffusion fluxes, predictor, PPE source, pressure
solve, corrector, face-velocity correction) of the channel workload on
resident device state.  Legs run the same steps from the same initial state
on one GPU, each at a pressure-solve tolerance eps (the reference's stopping
rule min(|r|_1/|b|_1, |r|_2/|b|_2) < eps):
  fp64     the reference's arithmetic (Jacobi-preconditioned BiCGSTAB in FP64);
  fp64_cg  single-reduction CG with the 4-layer block-Jacobi
           preconditioner in FP64 (separates the gain of a CG solver from
           the gain of FP32);
  mixed    the precision form: the solve by the vertical modes of the
           operator (NSX_REFINE_MODAL: per column the generalized
           eigenvectors of the vertical couplings split the PPE into one 2D
           problem per mode, each solved by FP64 CG with an FP32
           multigrid), in cycles from the true FP64 residual, stopped on it;
  mixed_block  the previous precision form: the single-reduction block-
           Jacobi CG of fp64_cg in FP32 with reliable updates;
  mixed_flux32  the mixed leg with the momentum fluxes and the Smagorinsky
           eddy viscosity in FP32 arithmetic too (its errors are reported;
           the gate is the mixed leg's);
  ref      fp64_cg at eps 1e-14, the tight reference the other legs'
           errors are measured against.
The precision-form legs (fp64_cg and the mixed ones) start each pressure
solve from 2 p_k - p_{k-1} of the same RK stage's last two solutions
(--guess extrapolate, NSX_GUESS_EXTRAPOLATE: about 5 % fewer iterations);
fp64 and ref start from the stage's input pressure, as the reference does
(--guess previous sets that for every leg).
The headline legs run at the gate tolerance (--eps-gate, 1e-13), where the
mixed leg's u, v, w and p agree with the FP64 leg's to the 1e-8 gate with
margin (at 1e-12 the pressures agree to 2.5e-9 to 2.7e-8 depending on the
step; at the workload's 1e-10 the FP64 BiCGSTAB's own pressure is 3e-6 from
the tight reference, the mixed leg's 2e-7).  The fp64 and mixed legs also
run at --eps-config (1e-10).  Each leg: W warm-up steps, K timed steps (wall
clock), then one step with HIP events around every solver kernel for the
per-kernel roofline.  Prints one JSON line:
  value        prism-cell-steps/s of the mixed leg at the gate tolerance
               = interior prisms x K / wall
  fp64, fp64_cg, mixed   the legs at the gate tolerance; mixed_over_fp64 and
               mixed_over_fp64_cg their ratios
  rel_err      relative L2 error of u, v, w, p (interior) of the mixed leg
               against the FP64 leg after the same steps, both legs' max
               |cell divergence| and CFL number (glob_cfl on the device);
               gate_passed: every field within 1e-8
  at_config_eps  the fp64 and mixed legs at the workload's 1e-10
  vs_ref       each leg's relative errors against the tight reference
  roofline     the dominant kernel of the mixed leg (its 2D solves together,
               a cycle as one launch): algorithmic bytes per launch / mean
               launch time (HIP events on the library's stream)
  cpu_baseline the oracle (CPU restatement of the reference, 1 core) on a
               bounded sample of the same workload, extrapolated per step;
               cpu_baseline_all_cores the same with the oracle's solver on
               OMP_NUM_THREADS threads
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "3d-channel-flow-code_amd"))

METRIC = "prism-cell-steps/s: mixed-prec vs FP64 GPU at ≤1e-8 rel err; % HBM peak"
HBM_PEAK_GBS = 8000.0
# algorithmic HBM bytes per interior prism of each BiCGSTAB kernel, in units of
# the vector width (8 B FP64, 4 B FP32): A reads rt,q,rhat, writes vt; B
# reads rt,vt, writes t; C reads x,rt,q,vt,t,rhat, writes x,rt,q
PHASE_UNITS = {"a": 4, "b": 3, "c": 9}
KERNEL_NAMES = {"a": "k_bicg_a", "b": "k_bicg_b", "c": "k_bicg_c"}
# workload tag used in file names of the profiles: quads in x, quads in y, layers
TAG = {0: "32x16x32", 1: "128x64x64", 2: "256x128x96", 3: "64x32x48", 4: "512x256x128"}
WORKLOAD = {
    0: "32x16 quads x 32 layers = 32,768 prisms, Re_tau 180, dt 1e-3",
    1: "128x64 quads x 64 layers = 1,048,576 prisms, Re_tau 180, dt 5e-4, jittered mesh",
    2: "256x128 quads x 96 layers = 6,291,456 prisms, Re_tau 395, dt 2.5e-4, jittered mesh",
    3: "64x32 quads x 48 layers = 196,608 prisms, Re_tau 180, dt 5e-4, jittered mesh",
    4: "512x256 quads x 128 layers = 33,554,432 prisms, Re_tau 590, dt 1e-4, jittered mesh",
}


def cpu_baseline(case, mean_iters: float, cap: int = 100, parallel: bool = False) -> dict:
    """One projection stage of the oracle on the full mesh with BiCGSTAB capped
    at `cap` iterations; the step time is extrapolated with the GPU's mean
    iteration count per solve (FP64 leg).  parallel: the oracle built with
    OpenMP (the solver's loops over OMP_NUM_THREADS threads; the rest of the
    stage, 3 % of the serial step, stays on one thread)."""
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import oracle

    O = oracle.Oracle(case, parallel=parallel)
    cores = O.threads()
    O.set_max_iters(cap)
    for n in ("uf", "vf", "wf", "pf"):
        O.state(n)[:] = O.state(n[0] + "fn")
    t0 = time.perf_counter()
    O.hydro()
    wall = time.perf_counter() - t0
    t = O.timers()
    its = max(O.solver_record()["iter"], 1)
    t_iter = t["solve"] / its
    t_rest = t["hydro"] - t["solve"]
    step_s = case.params.FinRK * (t_rest + mean_iters * t_iter)
    what = "1 thread" if not parallel else f"OpenMP, {cores} threads on the solver"
    return {"value": case.n_interior / step_s, "unit": "prism-cell-steps/s", "cores": cores, "kind": "port",
            "sample": (f"oracle (C restatement of the reference, {what}) on the full mesh: one projection stage "
                       f"with BiCGSTAB capped at {its} iterations ({wall:.1f} s); step time = "
                       f"{case.params.FinRK} x (non-solver {t_rest:.2f} s + {mean_iters:.0f} iterations x "
                       f"{t_iter * 1e3:.1f} ms) with the FP64 GPU leg's mean iteration count"),
            "s_per_step": step_s}


# the mixed forms (refinement, reliable-update delta): "mixed" the vertical-mode
# solve (delta unused); "mixed_block" the single-reduction FP32 CG with the 4-layer
# block-Jacobi preconditioner (the library's default), "mixed_line" the same
# with the line preconditioner (whole columns), "mixed_point" with point
# Jacobi; "mixed_cg2" the point-Jacobi CG in two kernels per iteration
MIXED_MODES = {"mixed": (7, 0.1), "mixed_block": (5, 0.1), "mixed_line": (6, 0.1), "mixed_point": (4, 0.1),
               "mixed_cg2": (3, 0.1), "mixed_flux32": (7, 0.1)}
# the FP32 CG kernels: W reads rt, p and writes w; X reads e, rt, p, w and
# writes e, rt, p (units of 4 B per interior prism; the few X launches that
# form a true FP64 residual move more)
CG_UNITS = {"w": 3, "x": 7}
# the single-reduction CG: one kernel per iteration reading and writing rt,
# om, sg (6 units), and every other iteration also reading the last u, p and
# e and writing p and e (11 units): 8.5 units a launch on average; its rare
# true-residual and product launches are counted with it
CGS_UNITS = 8.5
CGS_KERNEL = {4: "k_cgs<float, 0>", 5: "k_cgs<float, 1>", 6: "k_cgs<float, 2>"}


def modal_kernels(case) -> dict:
    """timer -> (kernel name, algorithmic bytes per launch) of the vertical-mode
    solve: the forward transform reads r and writes the modal right-hand
    sides; the backward one reads the modal solutions and reads and writes x;
    the true residual reads b and x and writes r (FP64, interior prisms).  The
    2D solves' time is that of a whole cycle (or the part of one that the host
    queued at once), their bytes those of one column in one iteration of one
    mode: the columns' vectors once per sweep at their stored width, the
    coarser levels and the graph left out"""
    n, nzi = case.n_interior, case.NZ - 2
    kt = (nzi + 15) // 16
    # output tiles a block forms: what of the table fits 160 KB of LDS beside
    # the partial sums, at most 8; 0 where not one does
    fits = min(8, (160 * 1024 - 256) // (kt * 2048))
    panels = (kt + max(1, fits) - 1) // max(1, fits)
    mt = (kt + panels - 1) // panels if fits else 0
    # node-major modal vectors where the 2D solves run batched (meshes of this
    # many columns have the three levels that takes)
    batched = case.N_CELL0 >= 24576 and 16 * kt <= 1024
    kind = "<%d, %s>" % (mt, "true" if batched else "false")
    # batched: the update 52, the four sweeps 60, restriction and prolongation
    # 12, the product 20; a block per mode: its FP64 vectors r, x and A p (the
    # FP32 ones lie in LDS, as far as they fit)
    mg = ("k_mb_* (2D solves of every mode)", 144) if batched else ("k_modal_2d", 64)
    return {"modal_fwd": ("k_modal_fwd" + kind, 16 * n), "modal_bwd": ("k_modal_bwd" + kind, 24 * n),
            "modal_spmv": ("k_modal_true", 24 * n), "modal_mg": mg}


def leg(case, name: str, steps: int, warmup: int, eps: float, max_iters=None, guess: int = 0) -> dict:
    """One leg: `name` is fp64 (BiCGSTAB), fp64_cg (FP64 single-reduction
    CG) or one of MIXED_MODES, with the pressure solves stopped at eps; guess
    is the initial-guess mode of the precision forms (0 the stage's input
    pressure, 1 extrapolated)."""
    from nsx.device import Context

    precision = {"fp64": 0, "fp64_cg": 2, "mixed_flux32": 3}.get(name, 1)
    ctx = Context(case)
    p = case.params
    ctx.set_params(eps=eps, max_iters=max_iters or p.MaxIters)
    if precision in (1, 3):
        ctx.set_precision(precision, *MIXED_MODES[name])
    if guess and precision != 0:
        ctx.set_initial_guess(guess)
    ctx.init_state()
    if warmup:
        ctx.step(warmup, precision)
    info0 = ctx.solve_info()
    t0 = time.perf_counter()
    info = ctx.step(steps, precision)
    wall = time.perf_counter() - t0
    solves = info["n_solves"] - info0["n_solves"]
    iters = info["iters_total"] - info0["iters_total"]
    # per-kernel times: one more step with HIP events around each solver kernel
    ctx.timing(True)
    ctx.timing_reset()
    ctx.step(1, precision)
    ctx.timing(False)
    n = case.n_interior
    kernels = {}
    for ph, units in PHASE_UNITS.items():
        ms, launches = ctx.timer("bicg_" + ph)
        if launches:
            avg = ms / launches
            b = units * 8 * n
            kernels["bicg_" + ph] = {"kernel": KERNEL_NAMES[ph] + "<double>", "launches": launches,
                                     "avg_us": avg * 1e3, "bytes_per_launch": b, "GBps": b / (avg * 1e-3) / 1e9}
    for ph, units in CG_UNITS.items():
        ms, launches = ctx.timer("cg32_" + ph)
        if launches:
            avg = ms / launches
            b = units * 4 * n
            kernels["cg32_" + ph] = {"kernel": "k_cg_" + ph, "launches": launches, "avg_us": avg * 1e3,
                                     "bytes_per_launch": b, "GBps": b / (avg * 1e-3) / 1e9}
    for tname, width in (("cg32_sr", 4), ("cg64_sr", 8)):
        ms, launches = ctx.timer(tname)
        if launches:
            avg = ms / launches
            b = int(CGS_UNITS * width * n)
            kname = "k_cgs<double, 1>" if width == 8 else CGS_KERNEL[MIXED_MODES[name][0]]
            kernels[tname] = {"kernel": kname, "launches": launches, "avg_us": avg * 1e3, "bytes_per_launch": b,
                              "GBps": b / (avg * 1e-3) / 1e9}
    for tname, (kname, b) in modal_kernels(case).items():
        ms, launches = ctx.timer(tname)
        if launches:
            avg = ms / launches
            if tname == "modal_mg":
                b = b * case.N_CELL0 * ctx.timer("modal_swept")[1] / launches
            kernels[tname] = {"kernel": kname, "launches": launches, "avg_us": avg * 1e3, "bytes_per_launch": b,
                              "GBps": b / (avg * 1e-3) / 1e9}
    stage_ms, stage_n = ctx.timer("stage")
    fields = {f: np.asarray(ctx.get(f))[:case.N_CELL0, 1:-1].copy() for f in ("UFN", "VFN", "WFN", "PFN")}
    # glob_cfl on the device: the largest net cell flux (cfl.F90:131-167) and the CFL number
    cfl = ctx.glob_cfl()
    fields["div"] = abs(cfl["flux_max"])
    fields["cfl"] = cfl["cfl"]
    ctx.close()
    return {"eps": eps, "value": n * steps / wall, "ms_per_step": wall / steps * 1e3, "wall": wall,
            "mean_iters_per_solve": iters / max(solves, 1), "solves": solves, "exit": info["exit"],
            "last_iters_fp32": info.get("iters_fp32", 0),
            "last_e1": info["e1"], "last_e2": info["e2"], "updates_last": info.get("outer_passes", 0),
            "kernels": kernels, "non_solver_ms_per_stage": stage_ms / max(stage_n, 1) * 2 if stage_n else None,
            "fields": fields}


def field_errors(fb: dict, fa: dict) -> dict:
    """relative L2 errors of u, v, w, p of leg b against leg a (interior prisms)"""
    err = {}
    for f, nm in (("UFN", "u"), ("VFN", "v"), ("WFN", "w"), ("PFN", "p")):
        err[nm] = float(np.linalg.norm(fb[f] - fa[f]) / max(np.linalg.norm(fa[f]), 1e-300))
    return err


def traffic_of(cfg: int, kernel):
    """HBM bytes per launch of `kernel` (fetch + write) from the committed
    rocprofv3 --pmc summary of this workload, or None"""
    if not kernel:
        return None
    from nsx.profsum import read_traffic

    t = read_traffic(os.path.join(REPO, "profiles", f"solver_traffic_channel_{TAG[cfg]}.txt"))
    key = kernel.replace(" ", "")
    if key not in t:
        return None
    return t[key][0] + t[key][1]


GATE = 1e-8


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=None)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--cfg", type=int, default=2)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--seed", type=int, default=1234)
    ap.add_argument("--eps-gate", type=float, default=1e-13,
                    help="pressure-solve tolerance of the headline legs (fp64, fp64_cg, mixed)")
    ap.add_argument("--eps-config", type=float, default=None,
                    help="the workload's own tolerance (default: the case's, 1e-10); 0 skips those legs")
    ap.add_argument("--eps-ref", type=float, default=1e-14, help="tolerance of the tight reference; 0 skips it")
    ap.add_argument("--legs", default="fp64,fp64_cg,mixed,mixed_block,mixed_flux32",
                    help="comma list of the gate legs: fp64, fp64_cg, mixed, mixed_block, mixed_flux32, mixed_line, "
                         "mixed_point, mixed_cg2")
    ap.add_argument("--max-iters", type=int, default=None,
                    help="cap the solver iterations (profiling runs only: the line is then marked capped)")
    ap.add_argument("--guess", choices=("extrapolate", "previous"), default="extrapolate",
                    help="initial guess of the precision-form legs' pressure solves")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="first copy one cell field with k_copy (the known-size copy for HBM counter calibration)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the multi-GPU sharding of the path is a design note, not code)", file=sys.stderr)
        return 2

    from nsx.case import config_case

    cfg = args.cfg
    steps = args.steps if args.steps is not None else {0: 10, 1: 20, 2: 10, 3: 20, 4: 3}[cfg]
    case = config_case(cfg, seed=args.seed)
    eps_cfg = case.params.eps if args.eps_config is None else args.eps_config
    legs = [x.strip() for x in args.legs.split(",") if x.strip()]
    if args.calibrate_copy:
        from nsx.device import Context
        c0 = Context(case)
        c0.copy(64, 0)  # CELL_SCRATCH <- UFN: N_CELL0 x NS doubles, NS = NZ rounded up to a multiple of 4
        c0.close()
        ns = (case.NZ + 3) // 4 * 4
        print(f"# k_copy calibration: {case.N_CELL0 * ns} doubles", file=sys.stderr, flush=True)

    guess = 1 if args.guess == "extrapolate" else 0

    def run(name, eps, g=None):
        r = leg(case, name, steps, args.warmup, eps, args.max_iters, guess if g is None else g)
        print(f"# leg {name} at eps {eps:g}: {r['value']:.4g} prism-cell-steps/s, {r['ms_per_step']:.1f} ms/step, "
              f"{r['mean_iters_per_solve']:.1f} iterations/solve", file=sys.stderr, flush=True)
        return r

    res = {name: run(name, args.eps_gate) for name in legs}
    at_cfg = {}
    if eps_cfg > 0 and eps_cfg != args.eps_gate:
        for name in ("fp64", "mixed"):
            if name in legs:
                at_cfg[name] = run(name, eps_cfg)
    ref = run("fp64_cg", args.eps_ref, 0) if args.eps_ref > 0 else None

    head = res.get("mixed") or res.get("fp64") or next(iter(res.values()))
    kern = head["kernels"]
    # the dominant kernel (of the mixed leg all 2D solves together): the most time
    dom_name = max(kern, key=lambda k: kern[k]["avg_us"] * kern[k]["launches"]) if kern else None
    dom = kern.get(dom_name, {"GBps": 0.0, "bytes_per_launch": 0, "avg_us": 0.0, "kernel": None})
    out = {
        "metric": METRIC,
        "value": head["value"],
        "unit": "prism-cell-steps/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": args.warmup,
        "ms_per_step": head["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": ("f64+f32 (FP64 CG per vertical mode, FP32 multigrid, MFMA FP64 transforms, FP64 true residuals)"
                  if "mixed" in res else ("f64" if "fp64" in res else "f32+f64")),
        "data": "synthetic",
        "config": {"workload": f"channel {WORKLOAD[cfg]}", "prisms": case.n_interior,
                   "time_scheme": "RK2 (FinRK=2)", "les": "Smagorinsky Cs=0.1", "ppe_tolerance": args.eps_gate,
                   "ppe_tolerance_workload": case.params.eps,
                   "ppe_solver": "vertical-mode solve: FP64 CG per mode with an FP32 smoothed-aggregation V-cycle, "
                                 "cycles from FP64 true residuals",
                   "initial_guess": {"precision_forms": args.guess, "fp64": "previous"},
                   "seed": args.seed},
        "roofline": {"bound": "hbm", "kernel": dom["kernel"], "achieved": dom["GBps"], "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": dom["GBps"] / HBM_PEAK_GBS, "traffic": traffic_of(cfg, dom["kernel"]),
                     "avg_launch_us": dom["avg_us"], "bytes_per_launch": dom["bytes_per_launch"]},
    }
    for name, r in res.items():
        out[name] = {k: v for k, v in r.items() if k != "fields"}
    if args.max_iters:
        out["capped_max_iters"] = args.max_iters

    def compare(rs, tag):
        """ratios and errors of the mixed forms against fp64 (and fp64_cg) within one set of legs"""
        o = {}
        for name in rs:
            if not name.startswith("mixed") or "fp64" not in rs:
                continue
            sfx = "" if name == "mixed" else name[5:]
            o["mixed_over_fp64" + sfx] = rs[name]["value"] / rs["fp64"]["value"]
            if "fp64_cg" in rs:
                o["mixed_over_fp64_cg" + sfx] = rs[name]["value"] / rs["fp64_cg"]["value"]
            fa, fb = rs["fp64"]["fields"], rs[name]["fields"]
            err = field_errors(fb, fa)
            err["max_div_fp64"] = fa["div"]
            err["max_div_mixed"] = fb["div"]
            err["cfl_fp64"] = fa["cfl"]
            err["cfl_mixed"] = fb["cfl"]
            err["gate"] = GATE
            err["gate_passed"] = bool(max(err["u"], err["v"], err["w"], err["p"]) <= GATE)
            o["rel_err" + sfx] = err
        if "fp64_cg" in rs and "fp64" in rs:
            o["fp64_cg_over_fp64"] = rs["fp64_cg"]["value"] / rs["fp64"]["value"]
        return o

    out.update(compare(res, "gate"))
    if at_cfg:
        sub = {"eps": eps_cfg}
        for name, r in at_cfg.items():
            sub[name] = {k: v for k, v in r.items() if k not in ("fields", "kernels")}
        sub.update(compare(at_cfg, "config"))
        out["at_config_eps"] = sub
    if ref is not None:
        vs = {"eps": args.eps_ref, "solver": "fp64_cg", "ms_per_step": ref["ms_per_step"],
              "mean_iters_per_solve": ref["mean_iters_per_solve"], "exit": ref["exit"]}
        for name, r in res.items():
            vs[f"{name}@{args.eps_gate:g}"] = field_errors(r["fields"], ref["fields"])
        for name, r in at_cfg.items():
            vs[f"{name}@{eps_cfg:g}"] = field_errors(r["fields"], ref["fields"])
        out["vs_ref"] = vs
    if not args.no_cpu:
        base = res.get("fp64", head)
        cb = cpu_baseline(case, base["mean_iters_per_solve"])
        out["cpu_baseline"] = {k: v for k, v in cb.items() if k != "s_per_step"}
        out["gpu_over_cpu"] = out["value"] / cb["value"]
        cbp = cpu_baseline(case, base["mean_iters_per_solve"], parallel=True)
        out["cpu_baseline_all_cores"] = {k: v for k, v in cbp.items() if k != "s_per_step"}
        out["gpu_over_cpu_all_cores"] = out["value"] / cbp["value"]
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
