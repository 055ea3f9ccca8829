#!/usr/bin/env python3
"""Throughput of the 3D smoke forward step on one MI355X.

Workload: 256^3 MAC grid, FP32, 500 steps from rest; velocity, density and temperature
advection; buoyancy (alpha 0.05, beta 0.5) and vorticity confinement (eps 0.3); attenuation
0.99 per step on velocity, temperature and density; mixed-precision red-black SOR projection
(FP32 sweeps, FP64 residual refinement) to max|div| <= 1e-6 on every step with a warm start,
omega 1.968 (the best of a sweep over 1.93-1.99 on this 500-step run; --omega overrides, --omega 0
takes Young's 2/(1+sin(pi/n))); MAC->regular output
every 10 steps.  Closed box (one-cell solid shell), sphere source of radius 0.08 at
(0.5, 0.1, 0.5) with density 1 and temperature 1, Tamb 0, seeded +-0.01 temperature noise,
dt 0.02, 20 advection substeps.  Inputs are resident in HBM before the timed region.  The
warm-up steps run first on the same simulation, whose state is then reset, so the timed region
is the workload's own steps 0..499; inside it only the sweep loops carry (pooled, unwaited) event
pairs, and the per-stage breakdown comes from a few event-timed steps after it.

fwd_adjoint: a 64-step window of the same workload, started from the state the timed steps
reached, run forward with a state checkpoint every 8 steps (sqrt of the window) and every step's
FP64 pressure kept, then through the hand-written adjoint (each earlier segment recomputed from its
checkpoint, replaying the kept pressures), for the loss 1/2 |rho_64 - target|^2 with a target of 8
seeded Gaussian blobs and per-step control forces (zero); value = voxels * window / (forward +
backward wall time).  without_pressure_store: the same window re-solving every recomputed step.

coarse_projection: the reference's default solver (COARSE_OPEN_POISSON_SOR) in a full step of its
expsimu3D/fine256.txt scene (256^3, 8^3 blocks, 600 coarse iterations, internal sphere, box
source), the scene parsed by the library's config reader; value = voxels * steps / wall time.

octree_projection: the same scene with globalGridSolver OPEN_OCTREE_POISSON_SOR (leaves of 1, 2^3,
4^3 and 8^3 cells from the distance to the sphere, thresholds 2/4/16, 600 red-black passes over
the levels); value = voxels * steps / wall time.

ensemble: 64 independent grids with per-axis sizes drawn from {32..96} (seeded, anisotropic),
alpha in [0.02, 0.1] and beta in [0.2, 1.0] per member, closed boxes with the same sphere
source, plain red-black SOR (omega 1.8, 200 iterations), 100 steps replayed from one captured
hipGraph after the launch-shape autotuner; value = all members' voxels * steps / wall time.

Prints one JSON line.  value = voxels * steps / wall time (Mvoxel-steps/s).  roofline: the
red-black SOR sweep kernel the autotuner picked (the dominant kernel), algorithmic bytes 13 B/voxel
per launch (a kernel that runs two iterations a launch reads and writes the grid once for both;
6.5 B/voxel for a single-colour launch) over its event-timed mean launch time; step_frac: the whole
step's algorithmic bytes over the step time.  cpu_baseline: the
CPU oracle on a bounded sample of the same step (see --help).
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
METRIC = "Mvoxel-steps/s at 256³ fwd & fwd+adjoint; HBM GB/s vs peak; divergence"
HBM_PEAK_GBS = 8000.0
SOR_BYTES_PER_VOXEL = 13.0  # of one pass of the sweeps over the grid
FULL_RUN = 500  # steps of the 256^3 workload
# SOR relaxation of the 256^3 workload: the best of 1.93, 1.95, 1.96, 1.965, 1.968, 1.97, 1.972, 1.98,
# 1.985, 1.99 over the 500-step run (sweeps per step 467, 334, 268, 235, 233, 237, 240, 325, 434, 635;
# Young's 1.9758: 282)
OMEGA = 1.968


def parse():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500,
                    help="timed steps, from the initial state (the workload runs 500; with fewer, the run "
                         "continues untimed to step 500 and the whole run is reported as full_run)")
    ap.add_argument("--warmup", type=int, default=5,
                    help="untimed steps first (the state is then reset to the initial one)")
    ap.add_argument("--size", type=int, default=256, help="grid edge (cube)")
    ap.add_argument("--inner", type=int, default=None,
                    help="FP32 SOR sweeps per refinement pass (at most, with --pass-rule 1 or 2); default 80, or "
                         "1000 with --pass-rule 2")
    ap.add_argument("--omega", type=float, default=OMEGA,
                    help="SOR relaxation (default %g, measured best on the 256^3 workload; 0: Young's "
                         "2/(1+sin(pi/n)) for the grid edge n)" % OMEGA)
    ap.add_argument("--full-run", type=int, default=FULL_RUN,
                    help="steps of the whole run: after the timed steps the run continues to this step on one clock "
                         "(reported as full_run; a value <= --steps adds nothing)")
    ap.add_argument("--profile-steps", type=int, default=10,
                    help="steps after the timed region run with per-stage event timing (the stage breakdown)")
    ap.add_argument("--max-outer", type=int, default=1000, help="refinement passes at most per step")
    ap.add_argument("--pass-rule", type=int, default=1, choices=(0, 1, 2),
                    help="refinement pass length (zq3d_sor_opts.pass_rule): 0 every pass runs --inner sweeps; "
                         "1 (default) fitted from the last pass's residual decay; 2 gated: a pass sweeps until an "
                         "iteration's largest update meets the tolerance (at most --inner sweeps)")
    ap.add_argument("--tol", type=float, default=1e-6, help="max|div| target")
    ap.add_argument("--warm-start", type=int, default=2, choices=(0, 1, 2),
                    help="projection start (zq3d_config.warm_start): 0 zero, 1 the previous step's pressure, "
                         "2 (default) extrapolated from the previous two steps' pressures")
    ap.add_argument("--warm-extrapolate", type=float, default=1.0,
                    help="with --warm-start 2: p1 + f (p1 - p2) (zq3d_config.warm_extrapolate; the library's "
                         "default is 0.5, steadier on start-up transients; on this workload 1 measured best)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--adj-window", type=int, default=64, help="steps of the forward+adjoint window (0: skip)")
    ap.add_argument("--ens-members", type=int, default=64, help="ensemble members (0: skip the ensemble leg)")
    ap.add_argument("--ens-steps", type=int, default=100, help="timed ensemble steps")
    ap.add_argument("--coarse-steps", type=int, default=5,
                    help="timed steps of the coarse + sub-grid projection leg (0: skip)")
    ap.add_argument("--octree-steps", type=int, default=3,
                    help="timed steps of the octree projection leg (0: skip)")
    ap.add_argument("--sor-shape", default=None,
                    help="sweep shape 'ty,zc' to use instead of autotuning it (a zq3d_autotune_sor candidate)")
    ap.add_argument("--traffic", default=None,
                    help="rocprofv3 FETCH_SIZE/WRITE_SIZE summary for the sweep kernel (default: "
                         "profiles/<kernel>_<W>_traffic.txt for the kernel the autotuner picked)")
    ap.add_argument("--cpu-c0", action="store_true",
                    help="also time the oracle on the whole 64^3 closed-box workload (100 steps, plain SOR omega "
                         "1.8 x 200) on one host thread and on all of them (about a minute)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="after the timed region run a plain 512 MiB device copy (3 launches) whose counter "
                         "readings scale FETCH_SIZE/WRITE_SIZE to bytes")
    args = ap.parse_args()
    if args.inner is None:
        args.inner = 1000 if args.pass_rule == 2 else 80
    return args


def make_state(W, H, D):
    from zq_smokesimulation_amd import noise_field
    occ = np.zeros((D, H, W), np.uint8)
    occ[0] = occ[-1] = 1
    occ[:, 0] = occ[:, -1] = 1
    occ[:, :, 0] = occ[:, :, -1] = 1
    T = noise_field(W, H, D, 0, 0.01)
    z = np.zeros
    return dict(u=z((D, H, W + 1), np.float32), v=z((D, H + 1, W), np.float32), w=z((D + 1, H, W), np.float32),
                T=T, rho=z((D, H, W), np.float32), occ=occ)


SOURCE = [0.5, 0.1, 0.5, 0.08, 1.0, 1.0]


def read_traffic(path):
    """FETCH_SIZE / WRITE_SIZE per dispatch (KiB) and the copy-kernel scale, from a profile summary."""
    if not os.path.exists(path):
        return None
    vals = {}
    for line in open(path):
        if ":" in line and not line.lstrip().startswith("#"):
            k, _, v = line.partition(":")
            words = v.split()
            if not words:
                continue
            try:
                vals[k.strip()] = float(words[0])
            except ValueError:
                vals[k.strip()] = words[0]
    need = ("kernel", "fetch_kib_per_dispatch", "write_kib_per_dispatch", "fetch_scale", "write_scale", "size")
    if not all(k in vals for k in need):
        return None
    return vals


def cpu_baseline(state, W, H, D, inner, sweeps_mean, omega):
    """The CPU oracle on a bounded sample of one step, on the GPU's own state:
    (1) a whole step whose projection stops after its first FP64 residual (no refinement pass),
    (2) `inner` red-black SOR iterations of the oracle on the same grid;
    step time = (1) + (GPU's mean sweeps per step) x (2) / inner.  The passes' residual/update work is
    left out, which favours the CPU slightly."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import zq_oracle as O
    p = dict(h=1.0 / W, dt=0.02, steps=20, Tamb=0.0, beta=0.5, alpha=0.05, eps=0.3, aV=0.99, aT=0.99, aR=0.99,
             adv_vel_type=0, adv_sca_type=2, open_mask=0, closed_mean=1, omega=omega, sor_iters=inner, mixed=1,
             max_outer=0, tol=0.0)
    s = {k: a.copy() for k, a in state.items()}
    t0 = time.perf_counter()
    O.step(p, s["u"], s["v"], s["w"], s["T"], s["rho"], s["occ"], p64=s["p64"], spheres=[SOURCE])
    t_fixed = time.perf_counter() - t0
    nc = O.sor_count(state["occ"], 0)
    rhs = O.divergence(state["u"], state["v"], state["w"], state["occ"])
    e = np.zeros((D + 2, H + 2, W + 2), np.float32)
    t0 = time.perf_counter()
    O.sor(nc, rhs, e, omega, inner)
    t_pass = time.perf_counter() - t0
    step_s = t_fixed + sweeps_mean * t_pass / inner
    return {
        "value": (W * H * D) / step_s / 1e6,
        "unit": "Mvoxel-steps/s",
        "cores": int(O.lib().orc_num_threads()),
        "kind": "port",
        "sample": ("oracle at %dx%dx%d on the GPU's state after the timed steps: one step with no refinement pass "
                   "(%.2f s) + %d SOR iterations (%.3f s); step time = %.2f + %.1f sweeps (GPU mean per step) x "
                   "%.3f / %d = %.2f s" % (W, H, D, t_fixed, inner, t_pass, t_fixed, sweeps_mean, t_pass, inner,
                                           step_s)),
    }


def cpu_c0():
    """The oracle on the whole 64^3 closed-box workload: closed walls, zero initial velocity, sphere
    source (r 0.08 at (0.5, 0.1, 0.5), density 1, temperature 1), seeded +-0.01 temperature noise,
    alpha 0.05, beta 0.5, eps 0.3, dt 0.02, 20 substeps, red-black SOR omega 1.8 x 200 with the
    closed-domain mean, 100 steps; timed on one thread and on every host thread."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import zq_oracle as O
    W = 64
    p = dict(h=1.0 / W, dt=0.02, steps=20, Tamb=0.0, beta=0.5, alpha=0.05, eps=0.3, aV=1.0, aT=1.0, aR=1.0,
             adv_vel_type=0, adv_sca_type=2, open_mask=0, closed_mean=1, omega=1.8, sor_iters=200, mixed=0,
             max_outer=0, tol=1e-6)
    out = {}
    for label, threads in (("one_thread", 1), ("all_threads", 0)):
        O.lib().orc_set_num_threads(threads)
        occ, u, v, w = O.init_fine_grid(W, W, W, O.ALL_FACES, 0)
        T = O.noise(W, W, W, 0, 0.01)
        R = np.zeros_like(T)
        t0 = time.perf_counter()
        for _ in range(100):
            O.step(p, u, v, w, T, R, occ, spheres=[SOURCE])
        wall = time.perf_counter() - t0
        out[label] = {"value": round(W ** 3 * 100 / wall / 1e6, 4), "unit": "Mvoxel-steps/s",
                      "cores": int(O.lib().orc_num_threads()), "seconds": round(wall, 2),
                      "density_total": float(R.astype(np.float64).sum())}
    O.lib().orc_set_num_threads(0)
    out["kind"] = "port"
    out["sample"] = "the whole 64^3 closed-box workload, 100 steps, plain SOR omega 1.8 x 200"
    return out


def ensemble_leg(args):
    """The batched-ensemble workload (see the module docstring)."""
    import zq_smokesimulation_amd as z
    from zq_smokesimulation_amd.ensemble import SmokeEnsemble, member_config
    rng = np.random.default_rng(0)
    cfgs, states = [], []
    for m in range(args.ens_members):
        W, H, D = (int(x) for x in rng.integers(32, 97, size=3))
        alpha, beta = float(rng.uniform(0.02, 0.1)), float(rng.uniform(0.2, 1.0))
        cfgs.append(member_config(W, H, D, voxel_size=1.0 / W, step_time=0.02, steps=20, Tamb=0.0, buoyancy=beta,
                                  gravity=alpha, confine=0.3, sor_open_mask=0, sor_closed_mean=1, sor_omega=1.8,
                                  sor_iters=200, sor_mixed_precision=0))
        st = make_state(W, H, D)
        st["T"] = z.noise_field(W, H, D, m, 0.01)
        states.append(st)
    ens = SmokeEnsemble(cfgs)
    for m, st in enumerate(states):
        ens.set_state(m, **st)
        ens.set_sources(m, spheres=[SOURCE])
    cells = ens.cells()
    ens.step(5, graph=False)
    ens.synchronize()
    t0 = time.perf_counter()
    ens.step(5, graph=False)
    ens.synchronize()
    eager = (time.perf_counter() - t0) / 5
    tune = ens.autotune(10)
    ens.step(1, graph=True)  # capture
    ens.synchronize()
    t0 = time.perf_counter()
    ens.step(args.ens_steps, graph=True)
    ens.synchronize()
    wall = time.perf_counter() - t0
    rho0 = ens.download(0, z._lib.FIELD_RHO)
    ens.close()
    sizes = [(c.width, c.height, c.depth) for c in cfgs]
    return {
        "value": round(cells * args.ens_steps / wall / 1e6, 3),
        "unit": "Mvoxel-steps/s",
        "members": len(cfgs),
        "cells": cells,
        "steps": args.ens_steps,
        "ms_per_step": round(1e3 * wall / args.ens_steps, 3),
        "ms_per_step_eager": round(1e3 * eager, 3),
        "sor_iterations": 200,
        "smallest": min(sizes, key=lambda t: t[0] * t[1] * t[2]),
        "largest": max(sizes, key=lambda t: t[0] * t[1] * t[2]),
        "autotune": tune["best"],
        "density_finite": bool(np.isfinite(rho0).all()),
    }


# the reference's fine256 scene (expsimu3D/fine256.txt) with its default solver, COARSE_OPEN_POISSON_SOR
FINE256 = ("resolution 256 256 256\nsubSize 8\nsource 0.5 0.1 0.5 0.1 0.05 0.1 0.8 20\nTamb 1\nconfineCoeff 30\n"
           "step 30\nstepTime 0.03\nframeCount 200\nmaxIter 600\ninnerIter 20\nvelAttenCoeff 10\n"
           "densityAttenCoeff 0\ntempAttenCoeff 0\nintObj sphere\nuseMovingObject false\n"
           "advVelType inReg_outReg\nadvScaType Reg\nexportType di3\naddForceType slice\n"
           "globalGridSolver COARSE_OPEN_POISSON_SOR\n")


def scene_leg(text, steps, warmup, workload):
    """A full step of a reference scene, parsed by the library's own config reader, timed over
    `steps` steps after `warmup`; returns the leg's record and the simulation's stage timing."""
    import tempfile
    import zq_smokesimulation_amd as z
    from zq_smokesimulation_amd import scene
    with tempfile.TemporaryDirectory() as td:
        path = os.path.join(td, "scene.txt")
        with open(path, "w") as f:
            f.write(text)
        sc = scene.load_scene(path)
        occ = scene.initial_occupancy(path)
    c = sc.config
    W, H, D = c.width, c.height, c.depth
    over = {n: getattr(c, n) for n, _ in c._fields_ if n not in ("struct_size", "width", "height", "depth", "sor")}
    over.update({"sor_" + n: getattr(c.sor, n) for n, _ in c.sor._fields_})
    over["octree_thresh"] = tuple(c.octree_thresh)
    sim = z.SmokeSim3D(W, H, D, **over)
    sweep = sim.coarse_sweep() if c.sub_size > 0 else None
    boxes = [list(sc.box_sources[i]) for i in range(sc.n_box_sources)]
    sim.set_box_sources(boxes)
    st = make_state(W, H, D)
    st["T"][...] = c.Tamb
    st["occ"] = occ
    sim.set_state(**st)
    for _ in range(warmup):
        sim.step()
    sim.synchronize()
    sim.set_profiling(True)
    stats = []
    t0 = time.perf_counter()
    for _ in range(steps):
        stats.append(sim.step())
    sim.synchronize()
    wall = time.perf_counter() - t0
    tm = sim.timing()
    rho = sim.download(z._lib.FIELD_RHO)
    sim.close()
    n = W * H * D
    rec = {
        "value": round(n * steps / wall / 1e6, 3),
        "unit": "Mvoxel-steps/s",
        "workload": workload,
        "steps": steps,
        "ms_per_step": round(1e3 * wall / steps, 3),
        "stages_ms_per_step": {k: round(tm[k] / max(tm["steps"], 1), 3) for k in
                               ("ms_force", "ms_advect_velocity", "ms_project", "ms_sor", "ms_advect_scalar",
                                "ms_reinject")},
        "max_div": float(max(s["max_div"] for s in stats)),
        "density_finite": bool(np.isfinite(rho).all()),
    }
    return rec, tm, sweep


def coarse_leg(args):
    """The reference's default projection (coarse + sub-grid, 8^3 blocks, 600 coarse iterations) in a
    full step of its fine256 scene."""
    rec, tm, sweep = scene_leg(FINE256, args.coarse_steps, args.warmup,
                               "expsimu3D/fine256.txt: 256^3, COARSE_OPEN_POISSON_SOR, subSize 8 (32^3 coarse "
                               "grid), maxIter 600, internal sphere, box source")
    # zc < 0: boxes held in registers, coded -(10000 log2(lx) + 100 ty + tz) threads
    rec["coarse_sweep_schedule"] = {"iterations_per_launch": sweep[0],
                                    "box" if sweep[1] < 0 else "planes_per_workgroup": sweep[1]}
    rec["coarse_sweep_launches_per_step"] = tm["sor_launches"] / max(tm["steps"], 1)
    return rec


def octree_leg(args):
    """The octree projection (OPEN_OCTREE_POISSON_SOR, octree_thresh 2/4/16, 600 passes over the four
    leaf levels) in a full step of the same fine256 scene."""
    text = FINE256.replace("globalGridSolver COARSE_OPEN_POISSON_SOR", "globalGridSolver OPEN_OCTREE_POISSON_SOR")
    rec, tm, _ = scene_leg(text, args.octree_steps, min(args.warmup, 3),
                           "expsimu3D/fine256.txt with globalGridSolver OPEN_OCTREE_POISSON_SOR: 256^3, leaves of "
                           "1, 2^3, 4^3, 8^3 cells (octree_thresh 2, 4, 16), maxIter 600, internal sphere, box source")
    launches = tm["sor_launches"] / max(tm["steps"], 1)
    rec["octree_sweep_launches_per_step"] = launches
    rec["octree_us_per_pass"] = round(1e3 * tm["ms_sor"] / max(tm["steps"], 1) / 600, 3)
    return rec


def adjoint_window(state, W, H, D, args, fwd_ms_per_step, shape, omega):
    """Forward + adjoint of a window of args.adj_window steps from `state` (FP32, sqrt(n) state
    checkpoints).  Run twice: without and then with the pressure store (every forward step's FP64
    pressure kept, so the recomputed steps replay it instead of solving again: the same states, the
    same gradient up to the order of the adjoint's atomic adds).  The record is the stored run, the
    plain one nested as without_pressure_store."""
    import math

    import torch
    from zq_smokesimulation_amd.adjoint import SmokeRollout
    from zq_smokesimulation_amd.gradcheck import gaussian_blobs
    n = args.adj_window
    K = max(1, int(round(math.sqrt(n))))
    eng = SmokeRollout(W, H, D, n, K, dtype=torch.float32, voxel_size=1.0 / W, step_time=0.02, steps=20, Tamb=0.0,
                       buoyancy=0.5, gravity=0.05, confine=0.3, vel_atten=0.99, temp_atten=0.99, dens_atten=0.99,
                       sor_open_mask=0, sor_closed_mean=1, sor_omega=omega, sor_iters=args.inner,
                       sor_max_outer=args.max_outer, sor_tol=args.tol, sor_pass_rule=args.pass_rule,
                       warm_start=1)
    if shape is not None:
        eng.set_sor_shape(shape["ty"], shape["zc"])
    eng.set_initial(**{k: torch.from_numpy(state[k]) for k in ("u", "v", "w", "T", "rho", "occ", "p64")})
    eng.set_sources(spheres=[SOURCE])
    target = torch.from_numpy(gaussian_blobs(W, H, D, 8, 0)).cuda()
    controls = torch.zeros(eng.controls_shape(), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    rho = eng.forward(controls)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    g = eng.backward(controls, rho - target)
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    fb, bb = eng.last_forward, eng.last_backward
    g = g.clone()
    gmax = float(g.abs().max())
    finite = bool(torch.isfinite(g).all())
    # the same window with every forward step's FP64 pressure kept: the recomputed steps apply the
    # forward's pressure instead of solving again (same states, same gradient up to atomic order)
    eng.set_pressure_store(True)
    torch.cuda.synchronize()
    s0 = time.perf_counter()
    rho2 = eng.forward(controls)
    torch.cuda.synchronize()
    s1 = time.perf_counter()
    g2 = eng.backward(controls, rho2 - target)
    torch.cuda.synchronize()
    s2 = time.perf_counter()
    bb2, fb2 = eng.last_backward, eng.last_forward
    eng.close()
    total, total2 = t2 - t0, s2 - s0
    plain = {
        "value": round(W * H * D * n / total / 1e6, 3),
        "ms_forward": round(1e3 * (t1 - t0), 1),
        "ms_backward": round(1e3 * (t2 - t1), 1),
        "ms_per_step": round(1e3 * total / n, 3),
        "ratio_to_window_forward": round(total / (t1 - t0), 3),
        "ratio_to_full_run_forward": round(1e3 * total / n / fwd_ms_per_step, 3),
        "recomputed_steps": bb["recomputed_steps"],
        "recompute_sweeps": bb["forward_sweeps"],
        "adjoint_sweeps_per_step": round(bb["adjoint_sweeps"] / n, 1),
    }
    return {
        "value": round(W * H * D * n / total2 / 1e6, 3),
        "unit": "Mvoxel-steps/s",
        "window": n,
        "checkpoint_every": K,
        "pressure_store": True,
        "ms_forward": round(1e3 * (s1 - s0), 1),
        "ms_backward": round(1e3 * (s2 - s1), 1),
        "ms_per_step": round(1e3 * total2 / n, 3),
        "ratio_to_window_forward": round(total2 / (s1 - s0), 3),
        "ratio_to_full_run_forward": round(1e3 * total2 / n / fwd_ms_per_step, 3),
        "recomputed_steps": bb2["recomputed_steps"],
        "recompute_sweeps": bb2["forward_sweeps"],
        "forward_sweeps_per_step": round(fb2["forward_sweeps"] / n, 1),
        "adjoint_sweeps_per_step": round(bb2["adjoint_sweeps"] / n, 1),
        "store_GB": round(n * (W + 2) * (H + 2) * (D + 2) * 8 / 1e9, 2),
        "max_div": max(fb["max_div"], fb2["max_div"]),
        "grad_max_abs": gmax,
        "grad_finite": finite and bool(torch.isfinite(g2).all()),
        "grad_max_diff_rel_vs_without_store": float((g2 - g).abs().max()) / max(gmax, 1e-30),
        "loss": "1/2 |rho_%d - target|^2, target = 8 seeded Gaussian blobs, controls = per-step cell forces" % n,
        "without_pressure_store": plain,
    }


def optimal_omega(n):
    """Young's optimal SOR relaxation for the 7-point Poisson operator on an n-cell edge:
    2 / (1 + sin(pi / n)) (the Jacobi iteration's spectral radius is cos(pi / n))."""
    import math
    return 2.0 / (1.0 + math.sin(math.pi / n))


def step_bytes(N, passes, residuals):
    """Algorithmic bytes of one forward step (compulsory reads and writes per stage, FP32 = 4 B,
    occupancy 1 B): force + attenuation 41, velocity advection 25, divergence 17, gradient correction
    29, scalar advection 29 (141 B/voxel), 13 B/voxel per pass of the SOR over the grid (one or
    more iterations) and 9 B/voxel per FP64 residual evaluation."""
    return N * (141.0 + SOR_BYTES_PER_VOXEL * passes + 9.0 * residuals)


def main():
    args = parse()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py measures one GPU: this build runs the smoke step on a single MI355X "
              "(multi-GPU sharding is a design note, not built); run with --gpus 1", file=sys.stderr)
        sys.exit(2)
    sys.path.insert(0, ROOT)
    import torch
    import zq_smokesimulation_amd as z

    W = H = D = args.size
    N = W * H * D
    omega = args.omega if args.omega > 0 else optimal_omega(max(W, H, D))
    sim = z.SmokeSim3D(W, H, D, voxel_size=1.0 / W, step_time=0.02, steps=20, Tamb=0.0, buoyancy=0.5, gravity=0.05,
                       confine=0.3, vel_atten=0.99, temp_atten=0.99, dens_atten=0.99, sor_open_mask=0,
                       sor_closed_mean=1, sor_omega=omega, sor_iters=args.inner, sor_mixed_precision=1,
                       sor_max_outer=args.max_outer, sor_tol=args.tol, sor_pass_rule=args.pass_rule,
                       warm_start=args.warm_start, warm_extrapolate=args.warm_extrapolate)
    sim.set_sphere_sources([SOURCE])
    st0 = make_state(W, H, D)
    p64_zero = np.zeros((D + 2, H + 2, W + 2), np.float64)

    def reset():
        sim.set_state(**st0)
        sim.upload(z._lib.FIELD_P64, p64_zero)  # cold start of the pressure warm start

    reset()
    print("bench: %d^3, omega %.4f, warmup %d, timed %d" % (W, omega, args.warmup, args.steps), file=sys.stderr,
          flush=True)
    for i in range(args.warmup):
        sim.step()
        if i % 10 == 0:
            sim.mac_to_regular()
    sim.synchronize()
    if args.sor_shape:
        ty, zc = (int(x) for x in args.sor_shape.split(","))
        sim.set_sor_shape(ty, zc)
        best = {"ty": ty, "zc": zc, "us_per_iter": None}
        print("bench: warmup done; sweep shape set to %s" % args.sor_shape, file=sys.stderr, flush=True)
    else:
        tune = sim.autotune_sor(20)
        best = tune["candidates"][tune["best"]] if tune["best"] >= 0 else None
        print("bench: warmup done; sweep tile autotune %s" % json.dumps(tune), file=sys.stderr, flush=True)
    # the timed region runs the workload's steps from its initial state; only the sweep loops carry
    # event pairs (pooled, read after the region), so the timing adds no synchronisation
    reset()
    sim.synchronize()
    sim.set_profiling(2)
    stats = []
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        stats.append(sim.step())
        if i % 10 == 0:
            sim.mac_to_regular()
        if (i + 1) % 100 == 0:
            print("bench: %d steps" % (i + 1), file=sys.stderr, flush=True)
    sim.synchronize()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    tm = sim.timing()
    sor_kernel = sim.sor_kernel()
    # the workload runs FULL_RUN steps: when fewer are timed above, the run continues to its end on the
    # same clock, so the whole run's rate is reported beside the timed window's
    full_stats = list(stats)
    sim.set_profiling(0)
    for i in range(args.steps, max(args.steps, args.full_run)):
        full_stats.append(sim.step())
        if i % 10 == 0:
            sim.mac_to_regular()
        if (i + 1) % 100 == 0:
            print("bench: %d steps" % (i + 1), file=sys.stderr, flush=True)
    sim.synchronize()
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    # stage breakdown: a few more steps with an event pair per stage (waited for), outside the region
    sim.set_profiling(1)
    for i in range(args.profile_steps):
        sim.step()
    sim.synchronize()
    tm_stages = sim.timing()
    sim.set_profiling(0)
    if args.calibrate_copy:
        a = torch.ones(128 << 20, dtype=torch.float32, device="cuda")
        bcopy = torch.empty_like(a)
        for _ in range(3):
            torch.mul(a, 1.0, out=bcopy)
        torch.cuda.synchronize()
        del a, bcopy
    wall = t1 - t0
    ms_per_step = 1e3 * wall / args.steps
    value = N * args.steps / wall / 1e6
    outer_mean = float(np.mean([s["outer"] for s in stats]))
    sweeps_mean = float(np.mean([s["sweeps"] for s in stats]))
    max_div = float(max(s["max_div"] for s in stats))
    converged = all(s["converged"] == 1 for s in stats)

    # a launch runs two iterations in one pass over the grid, or one, or one colour of one
    iters = float(sum(s["sweeps"] for s in stats))
    launches = max(tm["sor_launches"], 1)
    launch_ms = tm["ms_sor"] / launches
    grid_passes = min(1.0, launches / max(iters, 1.0))  # per iteration
    bytes_per_launch = SOR_BYTES_PER_VOXEL * N * grid_passes * iters / launches
    achieved = bytes_per_launch / (launch_ms * 1e-3) / 1e9
    step_gbs = step_bytes(N, grid_passes * sweeps_mean, outer_mean + 1.0) / (ms_per_step * 1e-3) / 1e9
    traffic = None
    tr = read_traffic(args.traffic or os.path.join(ROOT, "profiles", "%s_%d_traffic.txt" % (sor_kernel, W)))
    if tr and int(tr["size"]) == W and tr["kernel"] == sor_kernel:
        traffic = 1024.0 * (tr["fetch_kib_per_dispatch"] * tr["fetch_scale"] +
                            tr["write_kib_per_dispatch"] * tr["write_scale"])
    sw = np.array([s["sweeps"] for s in stats])
    nfull = len(full_stats)
    full_ms = 1e3 * (t2 - t0) / nfull
    full_sweeps = float(np.mean([s["sweeps"] for s in full_stats]))
    full_passes = float(np.mean([s["outer"] for s in full_stats]))
    full_run = {
        "steps": nfull,
        "value": round(N * nfull / (t2 - t0) / 1e6, 3),
        "ms_per_step": round(full_ms, 3),
        "sor_sweeps_per_step": full_sweeps,
        "sor_sweeps_percentiles": {str(q): float(np.percentile([s["sweeps"] for s in full_stats], q))
                                   for q in (0, 50, 90, 100)},
        "max_div": float(max(s["max_div"] for s in full_stats)),
        "every_step_within_tol": all(s["converged"] == 1 and s["max_div"] <= args.tol for s in full_stats),
        "step_frac": round(step_bytes(N, grid_passes * full_sweeps, full_passes + 1.0) / (full_ms * 1e-3) / 1e9 /
                           HBM_PEAK_GBS, 4),
        "note": "steps 0..%d of the workload from rest on one clock (the timed steps included)" % (nfull - 1),
    }
    out = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "Mvoxel-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": "3D smoke forward step, %d^3 MAC grid, closed box, mixed-precision red-black SOR to "
                        "max|div|<=%g, %d steps from rest" % (W, args.tol, args.steps),
            "grid": [W, H, D],
            "advection_substeps": 20,
            "sor_omega": round(omega, 6),
            "sor_omega_rule": ("2/(1+sin(pi/n)), n = %d" % max(W, H, D) if args.omega <= 0 else
                               "measured: best of 1.93-1.99 over the 500-step run" if args.omega == OMEGA else
                               "given"),
            "sor_sweeps_per_pass": args.inner,
            "sor_pass_rule": args.pass_rule,
            "warm_start": {0: "zero", 1: "previous pressure",
                           2: "p1 + %g (p1 - p2)" % args.warm_extrapolate}[args.warm_start],
            "sor_tile_autotuned": best,
            "parallelism": "single GPU",
        },
        "roofline": {
            "bound": "hbm",
            "kernel": sor_kernel,
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": traffic,
            "algorithmic_bytes_per_launch": bytes_per_launch,
            "mean_launch_us": round(launch_ms * 1e3, 3),
            "step_achieved": round(step_gbs, 1),
            "step_frac": round(step_gbs / HBM_PEAK_GBS, 4),
            "step_bytes": "N*(141 + 13*launch passes over the grid + 9*(refinement passes + 1)) per step, "
                          "means over the timed steps",
        },
        "projection": {
            "sor_sweeps_per_step": sweeps_mean,
            "sor_sweeps_percentiles": {str(q): float(np.percentile(sw, q)) for q in (0, 50, 90, 100)},
            "refinement_passes_per_step": outer_mean,
            "max_div": max_div,
            "every_step_within_tol": converged and max_div <= args.tol,
        },
        "stages_ms_per_step": {k: round(tm_stages[k] / max(tm_stages["steps"], 1), 3) for k in
                               ("ms_force", "ms_advect_velocity", "ms_project", "ms_sor", "ms_advect_scalar",
                                "ms_reinject")},
        "stages_note": "stage times from %d event-timed steps after the run" % args.profile_steps,
        "full_run": full_run,
    }
    g = sim.get_state()
    g["p64"] = sim.download(z._lib.FIELD_P64)
    sim.close()
    if args.adj_window > 0:
        print("bench: forward+adjoint window of %d steps" % args.adj_window, file=sys.stderr, flush=True)
        out["fwd_adjoint"] = adjoint_window(g, W, H, D, args, full_ms, best, omega)
    if args.ens_members > 0:
        print("bench: ensemble of %d grids" % args.ens_members, file=sys.stderr, flush=True)
        out["ensemble"] = ensemble_leg(args)
    if args.coarse_steps > 0:
        print("bench: coarse + sub-grid projection (fine256 scene)", file=sys.stderr, flush=True)
        out["coarse_projection"] = coarse_leg(args)
    if args.octree_steps > 0:
        print("bench: octree projection (fine256 scene)", file=sys.stderr, flush=True)
        out["octree_projection"] = octree_leg(args)
    if not args.no_cpu_baseline:
        print("bench: cpu baseline", file=sys.stderr, flush=True)
        out["cpu_baseline"] = cpu_baseline(g, W, H, D, 40, sweeps_mean, omega)
    else:
        out["cpu_baseline"] = None
    if args.cpu_c0:
        print("bench: cpu baseline, 64^3 workload", file=sys.stderr, flush=True)
        out["cpu_baseline_64"] = cpu_c0()
    print(json.dumps(out))


if __name__ == "__main__":
    main()
