#!/usr/bin/env python
"""Benchmark of the MI355X fractional step on the 2048^2 lid-driven cavity.

Workload (the one the headline metric is quoted on): unit-square cavity,
2048 x 2048 cells, Re = 5000, lid u = 1, seeded divergence-free start, cfl 0.5
(dt = 0.5 / (4 n^2)), momentum tolerance 1e-10, Poisson tolerance 1e-10.

A "step" is one full time step (pseudo-iterations of the momentum predictor to
convergence, Poisson RHS, multigrid projection, update) over the whole grid.
The state is resident in HBM before the timed region; W warm-up steps run
first, then exactly K steps are timed between device synchronisations.

Both precisions are run from the same initial state:
  * mixed  -- FP32 stencils and FP32 V-cycle inside FP64 iterative refinement
              (the headline `value`)
  * fp64   -- the plain FP64 step
and the mixed result is compared with the FP64 one per field after the same
number of steps.  Beside them, two more legs are timed: the discrete adjoint
of a 512^2, Re = 1000 rollout (backward sweep with checkpoint recomputation
over the forward time), the two-level composite step (512^2 coarse level +
a ratio-2 patch over the top quarter) and the 3D step of the general path
(256^3 cavity, FP64).  One JSON line is printed.

roofline: after the timed steps of each precision, the same run advances K
more steps with the library's in-step kernel timing on (HIP events, created
without a system-scope fence, around each launch of the step's main kernels on
the library's stream; launches that exited at once past convergence are not
counted).  achieved = the kernel's algorithmic bytes per launch / its average
launch time there; `roofline` is the kernel of the headline run with the most
time per step, `kernel_rooflines` lists every timed kernel.  The events cost a
few per cent of the step time, so `value` comes from the first timed pass,
which runs without them.  traffic: rocprofv3 FETCH_SIZE + WRITE_SIZE per launch
from profiles/pmc_summary.txt, scaled by a 64 MiB copy.
fp64_step_roofline: algorithmic bytes of a whole FP64 step (model in
step_bytes_fp64) over the measured step time.
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK = 8.0e12  # MI355X HBM3E, bytes/s
# timing kinds of amressif_time_kernel (--kernel-probe) -> kernel symbol
KERNELS = {0: "amr::k_stage64<0, true> (FP64 stage)", 1: "amr::k_gsrb2<T, 1, R> (finest down-leg smoother + restriction)",
           3: "amr::k_stage64<3, true> (mixed residual)", 4: "amr::k_tangent",
           5: "amr::k_gsrb2<T, 2, R> (finest up-leg smoother + FP64 outer step)",
           6: "amr::k_stage_pair<false> (two FP64 stages, one pass)",
           10: "amr::k_mixed_pair (mixed iteration, one pass)"}
# in-step timed kernels (amressif_kernel_time) -> kernel symbol, key in profiles/pmc_summary.txt
STEP_KERNELS = {
    "stage": ("amr::k_stage64<0, true> (FP64 RK stage)", "stage_fp64"),
    "stage_last": ("amr::k_stage64<1, true> (FP64 last RK stage + norm partials)", None),
    "resid": ("amr::k_stage64<3, true> (mixed FP64 residual)", "residual_mixed"),
    "tangent": ("amr::k_tangent (mixed FP32 tangent-linear update)", "tangent_mixed"),
    "mg_down": ("finest down-leg smoother + restriction (amr::k_gsrb2<T, 1, 8, false, HS>)", "smooth1_{prec}"),
    "mg_up": ("finest up-leg smoother + FP64 outer step (amr::k_gsrb2<float, 2, 8, true, 6> mixed, "
              "amr::k_gsrb<double, 2, 8> FP64)", "smooth5_{prec}"),
    "project": ("amr::k_project (update + next step's BDF2 constant)", None),
    "poisson_start": ("amr::k_poisson_start (Poisson RHS, warm start, first residual)", None),
    "pair": ("amr::k_stage_pair<false> (FP64 RK stages 1-2 in one pass)", "pair_fp64"),
    "pair_last": ("amr::k_stage_pair<true> (FP64 RK stages 3-4 in one pass + norm partials)", None),
    "mpair": ("amr::k_mixed_pair (mixed residual + FP32 tangent-linear update in one pass)", "mpair_mixed"),
    "iter": ("amr::k_iter_tile (FP64 pseudo-iteration of four RK stages in one pass)", None),
}


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--n", type=int, default=2048)
    ap.add_argument("--ren", type=float, default=5000.0)
    ap.add_argument("--cpu-steps", type=int, default=3, help="oracle steps timed for cpu_baseline (0: skip)")
    ap.add_argument("--only", choices=["both", "mixed", "fp64"], default="both")
    ap.add_argument("--profile-run", action="store_true", help="short run for rocprofv3: no cpu baseline")
    ap.add_argument("--adjoint-n", type=int, default=512, help="adjoint leg grid (0: skip the leg)")
    ap.add_argument("--adjoint-steps", type=int, default=1000)
    ap.add_argument("--adjoint-every", type=int, default=32, help="checkpoint interval of the adjoint leg")
    ap.add_argument("--amr-n", type=int, default=512, help="two-level leg: coarse grid (0: skip the leg)")
    ap.add_argument("--amr-steps", type=int, default=500)
    ap.add_argument("--gen-n", type=int, default=256, help="3D leg: cells per side of the 3D cavity (0: skip)")
    ap.add_argument("--gen-steps", type=int, default=5)
    ap.add_argument("--kernel-probe", choices=["fp64", "mixed"], default=None,
                    help="for rocprofv3 --pmc: one step, then a few timed launches of each kernel of that "
                         "precision and a 64 MiB copy (calibration); prints their HIP-event times")
    return ap.parse_args()


def read_traffic(kernel_key: str):
    """HBM bytes per launch from the committed rocprofv3 --pmc summary, scaled by
    the copy-kernel calibration recorded next to it (None if absent)."""
    path = os.path.join(ROOT, "profiles", "pmc_summary.txt")
    if not os.path.exists(path):
        return None
    vals = {}
    for line in open(path):
        m = re.match(r"\s*([A-Za-z0-9_.]+)\s*:\s*([-+0-9.eE]+)\s*$", line)
        if m:
            vals[m.group(1)] = float(m.group(2))
    key = f"{kernel_key}.traffic_bytes"
    return vals.get(key)


def step_bytes_fp64(n, pseudo_iters, vcycles, pseudo_bytes=4 * 64):
    """Algorithmic HBM bytes of one FP64 step at n^2 cells, kernel by kernel:
    `pseudo_bytes` per cell and pseudo-iteration (four passes of 64 B, one per RK4
    stage; two, the first stage of each kept in registers; one of 48 B; the pressure
    gradient sits in the BDF2 constant, put there by the previous projection); per V-cycle the
    finest down-leg smoother with the fused restriction (r in, e out, coarse
    r out: 18 B), the finest up-leg smoother with the fused FP64 outer step
    (e, r, coarse e, phi, b in; phi, next r out: 50 B) and the coarser levels
    (down 18 B + up 26 B per cell of the level: 44/3 B per finest cell over the
    hierarchy; the single-workgroup tail is negligible); once per step the
    Poisson start (u*, v* in; b, phi0, r0 out: 40 B) and the projection with
    the next step's BDF2 constant (u*, v*, phi, p, u^n in; u, v, p, c and the
    copy of u out: 104 B)."""
    cells = float(n) * n
    return cells * (pseudo_iters * pseudo_bytes + vcycles * (18 + 50 + 44 / 3) + 40 + 104)


def run_precision(api, W, n, ren, precision, state, warmup, steps, torch):
    inp = api.cavity_inputs(n, ren, precision=precision)
    run = api.Run.from_numpy(inp, state)
    if warmup:
        run.advance(warmup)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    stats = run.advance(steps)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    return run, stats, t1 - t0


def in_step_kernels(run, steps, prec_name, n, torch):
    """Second timed pass of `steps` steps with per-launch HIP events: one
    roofline entry per kernel that ran, with its launches per step."""
    run.ctx.kernel_timing(True)
    run.advance(steps)
    torch.cuda.synchronize()
    run.ctx.kernel_timing(False)
    rows = []
    for key, (ms, cnt, nbytes) in run.ctx.kernel_times().items():
        if cnt == 0:
            continue
        sym, pmc = STEP_KERNELS[key]
        achieved = nbytes / (ms * 1e-3)
        rows.append({"bound": "hbm", "achieved": achieved / 1e9, "peak": HBM_PEAK / 1e9, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK,
                     "traffic": read_traffic(f"{pmc.format(prec=prec_name)}_{n}") if pmc else None,
                     "kernel": sym, "avg_launch_ms": ms, "algorithmic_bytes_per_launch": nbytes,
                     "launches_per_step": cnt / steps, "ms_per_step": ms * cnt / steps,
                     "timed": f"in-step, HIP events around each launch, {steps} steps"})
    return rows


def adjoint_leg(api, W, n, steps, every, torch):
    """Lid-and-initial-velocity gradient of the lower-left kinetic energy after
    `steps` FP64 steps (512^2, Re = 1000 by default): forward with checkpoints
    every `every` steps, then the backward sweep (segment recomputation + adjoint)."""
    from amressif_amd.adjoint import CheckpointedRollout, kinetic_energy_lower_left
    inp = api.cavity_inputs(n, 1000.0)
    ro = CheckpointedRollout(inp, steps, every=every)
    lid = torch.tensor(W.lid_profile(n), device="cuda")
    st = W.initial_state(n, "seeded")
    u0, v0 = torch.tensor(st["u"], device="cuda"), torch.tensor(st["v"], device="cuda")
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    u, v = ro.forward(lid, u0, v0)
    torch.cuda.synchronize()
    t_fwd = time.perf_counter() - t0
    u.requires_grad_(True)
    v.requires_grad_(True)
    J = kinetic_energy_lower_left(u, v)
    gu, gv = torch.autograd.grad(J, (u, v))
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    glid, gu0, gv0 = ro.backward(gu, gv)
    torch.cuda.synchronize()
    t_bwd = time.perf_counter() - t0
    import numpy as np
    return {"workload": f"lid-driven cavity {n}x{n}, Re=1000, seeded start + seeded lid profile, {steps} FP64 "
                        f"steps, J = lower-left kinetic energy, checkpoints every {every} steps",
            "forward_s": t_fwd, "backward_s": t_bwd, "ratio": t_bwd / t_fwd, "J": float(J.detach()),
            "grad_lid_norm": float(glid.norm()), "grad_u0_norm": float(torch.sqrt((gu0 ** 2).sum() + (gv0 ** 2).sum())),
            "mean_pseudo_iters": float(np.mean([s["pseudo_iters"] for s in ro.fwd_stats])),
            "mean_adjoint_sweeps": float(np.mean([s["lin_iters"] for s in ro.bwd_stats])),
            "adjoint_flags": int(np.bitwise_or.reduce([s["flags"] for s in ro.bwd_stats]))}


def amr_leg(api, W, n0, steps, torch):
    """Two-level forward step, mixed precision: coarse n0^2, ratio-2 patch over
    the top quarter (coarse rows [3 n0 / 4, n0)), Re = 2000, seeded field."""
    import numpy as np
    jc0 = 3 * n0 // 4
    inp = api.cavity_inputs(n0, 2000.0, precision=api.AMRESSIF_MIXED)
    tl = api.TwoLevel(inp, jc0, W.seeded_two_level(n0, jc0))
    tl.advance(2)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    st = tl.advance(steps)
    torch.cuda.synchronize()
    sec = time.perf_counter() - t0
    cells = n0 * jc0 + (2 * n0) * (2 * (n0 - jc0))
    return {"workload": f"two-level cavity: coarse {n0}x{n0} + ratio-2 patch {2 * n0}x{2 * (n0 - jc0)} over the top "
                        f"quarter, Re=2000, seeded start, mixed precision, composite FGMRES projection, {steps} steps",
            "composite_cells": cells, "mcell_steps_per_s": cells * steps / sec / 1e6, "ms_per_step": 1e3 * sec / steps,
            "mean_coarse_iters": float(np.mean([x["coarse_iters"] for x in st])),
            "mean_fine_iters": float(np.mean([x["fine_iters"] for x in st])),
            "mean_poisson_iters": float(np.mean([x["poisson_iters"] for x in st])),
            "max_div_ratio": float(max(x["div_new"] / max(x["div_star"], 1e-300) for x in st)),
            "flags": int(np.bitwise_or.reduce([x["flags"] for x in st]))}


def general_leg(api, n, steps, torch):
    """The general path on a 3D lid-driven cavity: n^3 cells, walls 135 with the
    lid (165, u = 1) on the y-hi side, Re = 1000, FP64, from rest after two
    warm-up steps; plus the rates of the cell-velocity pass and of the stage kernel."""
    import numpy as np
    inp = api.default_inputs(n_cell=n, max_grid_size=(n, n, n), IterNum=100, cfl=0.5, ren=1000.0, vis=1e-3,
                             phy_bc_lo=(135, 135, 135), phy_bc_hi=(135, 165, 135), inflow_waveform=(1.0, 0.0, 0.0),
                             momentum_tolerance=1e-10, spacedim=3)
    ctx = api.Context(inp)
    ctx.init_state()
    ctx.advance(2)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    st = ctx.advance(steps)
    torch.cuda.synchronize()
    sec = time.perf_counter() - t0
    names = {7: "amr::gen::k_gen_cells (cell velocities with ghosts)",
             8: "amr::gen::k_gen_stage3 (one RK4 stage)",
             9: "amr::gen::k_gen_stage3 (one RK4 stage + norm partials)"}
    kern = []
    for which, name in names.items():
        ms, nbytes = ctx.time_kernel(which, reps=10)
        kern.append({"kernel": name, "avg_launch_ms": ms, "algorithmic_bytes_per_launch": nbytes,
                     "achieved": nbytes / (ms * 1e-3) / 1e9, "unit": "GB/s", "frac": nbytes / (ms * 1e-3) / HBM_PEAK})
    return {"workload": f"3D lid-driven cavity {n}^3, Re=1000, from rest, FP64, tol 1e-10, {steps} steps",
            "mcell_steps_per_s": n ** 3 * steps / sec / 1e6, "ms_per_step": 1e3 * sec / steps,
            "mean_pseudo_iters": float(np.mean([s["pseudo_iters"] for s in st])),
            "mean_vcycles": float(np.mean([s["vcycles"] for s in st])),
            "flags": int(np.bitwise_or.reduce([s["flags"] for s in st])), "stage_kernels": kern}


def kernel_probe(api, W, n, ren, which_prec):
    """Isolated launches for the counter runs (rocprofv3 --pmc): one step,
    then a few timed launches of each kernel and a 64 MiB copy."""
    prec = api.AMRESSIF_MIXED if which_prec == "mixed" else api.AMRESSIF_FP64
    run = api.Run.from_numpy(api.cavity_inputs(n, ren, precision=prec), W.initial_state(n, "seeded"))
    run.advance(1)
    kinds = (10, 3, 4, 1, 5) if which_prec == "mixed" else (0, 6, 1, 5)
    res = {KERNELS[k]: run.ctx.time_kernel(k, reps=3)[0] for k in kinds}
    res["copy 64 MiB"] = run.ctx.time_kernel(2, reps=3, copy_bytes=64 << 20)[0]
    print(json.dumps({"kernel_probe": which_prec, "n": n, "avg_ms": res}), flush=True)


def main():
    args = parse()
    if args.gpus != 1:
        sys.stderr.write("bench.py: the library runs on one GPU only (the step is measured on one MI355X); "
                         f"--gpus {args.gpus} is not supported\n")
        sys.exit(2)
    import numpy as np
    import torch
    from amressif_amd import api
    from amressif_amd import workloads as W

    if args.kernel_probe:
        kernel_probe(api, W, args.n, args.ren, args.kernel_probe)
        return

    n, ren, K, Wu = args.n, args.ren, args.steps, args.warmup
    state = W.initial_state(n, "seeded")
    out = {}
    runs = {}
    for name, prec in (("mixed", api.AMRESSIF_MIXED), ("fp64", api.AMRESSIF_FP64)):
        if args.only not in ("both", name):
            continue
        run, stats, sec = run_precision(api, W, n, ren, prec, state, Wu, K, torch)
        P = float(np.mean([s["pseudo_iters"] for s in stats]))
        V = float(np.mean([s["vcycles"] for s in stats]))
        flags = int(np.bitwise_or.reduce([s["flags"] for s in stats]))
        worst_div = max(s["div_new"] / max(s["div_star"], 1e-300) for s in stats)
        out[name] = dict(mcell_steps_per_s=n * n * K / sec / 1e6, ms_per_step=1e3 * sec / K, pseudo_iters=P,
                         vcycles=V, flags=flags, max_div_ratio=worst_div)
        runs[name] = run
    # per-field error of mixed vs FP64: both runs have advanced W + K steps here
    fetched = {name: runs[name].fetch() for name in runs} if len(runs) == 2 else {}
    kernels = {name: in_step_kernels(runs[name], K, name, n, torch) for name in runs}

    # per-field error of mixed vs FP64 after the same W+K steps
    err = None
    if fetched:
        a, b = fetched["mixed"], fetched["fp64"]

        def rel(x, y):
            return float(np.abs(x - y).max() / max(np.abs(y).max(), 1e-300))

        pa, pb = a["ctx"][0, 1:-1, 1:-1], b["ctx"][0, 1:-1, 1:-1]
        fa, fb = a["ctx"][1, 1:-1, 1:-1], b["ctx"][1, 1:-1, 1:-1]
        err = {"U": rel(a["u"], b["u"]), "V": rel(a["v"], b["v"]),
               "p": rel(pa - pa.mean(), pb - pb.mean()), "phi": rel(fa - fa.mean(), fb - fb.mean())}

    # roofline of the headline run's dominant kernel: the one with the most
    # time per step in the in-step timed pass
    head = "mixed" if "mixed" in runs else "fp64"
    roofline = dict(max(kernels[head], key=lambda r: r["ms_per_step"]))
    extra = {f"{name}_kernels": kernels[name] for name in runs}
    if "fp64" in out:
        o = out["fp64"]
        sec = o["ms_per_step"] * 1e-3
        nbytes = step_bytes_fp64(n, o["pseudo_iters"], o["vcycles"])
        ran = [r["kernel"] for r in kernels.get("fp64", [])]
        per_iter, model = 4 * 64, "as above"
        if any(k.startswith("amr::k_stage_pair") for k in ran):
            per_iter, model = 2 * 64, ("two passes of 64 B/cell per pseudo-iteration (k_stage_pair: the first stage "
                                       "of each pair stays in registers)")
        elif any(k.startswith("amr::k_iter_tile") for k in ran):
            per_iter, model = 48, "one pass of 48 B/cell per pseudo-iteration (k_iter_tile: all four stages in registers)"
        nb2 = step_bytes_fp64(n, o["pseudo_iters"], o["vcycles"], per_iter)
        extra["fp64_step_roofline"] = {
            "bytes_per_step": nbytes, "achieved": nbytes / sec / 1e9, "unit": "GB/s", "frac": nbytes / sec / HBM_PEAK,
            "byte_model": "four RK4 stage passes of 64 B/cell per pseudo-iteration (the minimum traffic of "
                          "one-stage-per-pass kernels)",
            "bytes_per_step_as_run": nb2, "achieved_as_run": nb2 / sec / 1e9, "frac_as_run": nb2 / sec / HBM_PEAK,
            "byte_model_as_run": model}

    adj = None
    if args.adjoint_n > 0 and not args.profile_run:
        adj = adjoint_leg(api, W, args.adjoint_n, args.adjoint_steps, args.adjoint_every, torch)

    amr = None
    if args.amr_n > 0 and not args.profile_run:
        amr = amr_leg(api, W, args.amr_n, args.amr_steps, torch)

    gen = None
    if args.gen_n > 0 and not args.profile_run:
        gen = general_leg(api, args.gen_n, args.gen_steps, torch)

    cpu = None
    if args.cpu_steps > 0 and not args.profile_run:
        from oracle.refcpu import Oracle
        threads = int(os.environ.get("OMP_NUM_THREADS", "0")) or os.cpu_count()
        o = Oracle(n, ren, W.dt_from_cfl(n, 0.5), nthreads=threads)
        st = W.initial_state(n, "seeded")
        t0 = time.perf_counter()
        o.advance(st, args.cpu_steps)
        sec = time.perf_counter() - t0
        cpu = {"value": n * n * args.cpu_steps / sec / 1e6, "unit": "Mcell-steps/s", "cores": threads,
               "kind": "port",
               "sample": f"oracle/refcpu.c FP64 (MG Poisson), first {args.cpu_steps} steps of the same "
                         f"{n}^2 Re={ren:g} seeded workload, {threads} OpenMP threads, {sec:.1f} s"}

    value = out[head]["mcell_steps_per_s"]
    line = {
        "metric": "Mcell-steps/s 2048² mixed vs FP64 (err≤1e-6); adjoint:forward time ratio",
        "value": value,
        "unit": "Mcell-steps/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": Wu,
        "ms_per_step": out[head]["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32+f64" if head == "mixed" else "f64",
        "data": "synthetic",
        "config": {"workload": f"lid-driven cavity {n}x{n}, Re={ren:g}, seeded divergence-free start, "
                               f"cfl 0.5, tol 1e-10, {head} precision", "n_cell": n, "ren": ren,
                   "precision": head},
        "runs": out,
        "mixed_vs_fp64_speedup": (out["mixed"]["mcell_steps_per_s"] / out["fp64"]["mcell_steps_per_s"]
                                  if "mixed" in out and "fp64" in out else None),
        "mixed_vs_fp64_rel_err": err,
        "mixed_vs_fp64_rel_err_note": ("U, V and mean-removed p meet the 1e-6 bar; phi, the last step's pressure "
                                       "increment (about 1e-5 of p), follows where the momentum predictor stopped "
                                       "(momentum_tolerance 1e-10): two FP64 runs at momentum tolerances 1e-10 and "
                                       "1e-12 differ in phi by the same 1.7e-5, and with both runs at 1e-12 mixed "
                                       "and FP64 agree in phi to 8.4e-7 (tests/test_gpu_workloads.py)"),
        "adjoint_forward_ratio": adj["ratio"] if adj else None,
        "adjoint": adj,
        "two_level": amr,
        "general_3d": gen,
        "roofline": roofline,
        "kernel_rooflines": extra,
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
