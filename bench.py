#!/usr/bin/env python3
"""Throughput benchmark of the rigid-body step on one MI355X.

Headline workload (default): the sparse 1M-body scene — 1,000,000 spheres and
boxes (50/50, sizes U(0.25, 0.75) m) on a jittered 4 m lattice filling a 400 m
cube above the ground plane, about 2 % of bodies starting in contact, dt =
1/120 s — with every step's sweeps run until the contact residual is <= 1e-4
(checked inside the sweep launch after every sweep, at most 300 sweeps).  A
"step" is one full physics step (broadphase, narrowphase, colouring, solve to
the tolerance, integration) of the whole scene with its state resident in HBM.
The scene runs its 120 steps: 10 warm-up steps, then 110 timed steps replayed
from hipGraphs.

Prints one JSON line: body-steps/s at the tolerance and the fraction of steps
that reached it, the roofline of the dominant part of the solver's sweeps (240 B
per contact point per sweep, divided by the event-timed durations of its
launches) and of the whole step (304 N + 104 P + 304 C + 12 R C +
240 I C bytes per step), the energy drift of one step against an FP64 CPU
re-solve of the same manifolds, and the CPU oracle on the same workload (one
thread and all host cores).  Further sections: the dense 100k-body pile at its
fixed 20 sweeps over the configuration's 600 steps, and the plain vs learned
warm start at residual <= 1e-4.
"""
import argparse
import json
import os
import platform
import sys
import tempfile
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "axiom-physics-engine_amd"))

import numpy as np  # noqa: E402

import axm  # noqa: E402

HBM_PEAK_GBS = 8000.0
SEED_BASE = 0x4158494F4D000000
DT = 1.0 / 120.0
WORKLOADS = {
    0: "mixed spheres/boxes, 1k bodies, ground plane",
    1: "dense stacking pile: 100k spheres/boxes/capsules, 20x20 m footprint, 4 walls + ground",
    2: "sparse 1M spheres/boxes in a 400 m cube above the ground",
    3: "4096 independent worlds, 16-4096 bodies each",
}
DEFAULT_ITERS = {0: 10, 1: 20, 2: 10, 3: 10}
# algorithmic bytes (per body, pair, contact point, contact x colouring round, contact x sweep)
B_BODY, B_PAIR, B_CONTACT, B_ROUND, B_SWEEP = 304, 104, 304, 12, 240


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def host_cpu():
    model = platform.processor() or "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    nproc = os.cpu_count() or 1
    try:
        nproc = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        pass
    return model, nproc


def oracle_rate(desc, state, tol, max_sweeps, every, iters, threads, budget_s, fp64=False):
    """Steps the CPU oracle from `state` with the same solver settings (residual-stopped when tol > 0)
    for about budget_s seconds; returns (body-steps/s, steps, seconds, mean sweeps)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import orc

    ow = orc.OracleWorld(orc.params_from_desc(desc), fp64=fp64)
    ow.set_bodies(state)
    ow.set_threads(threads)
    if tol > 0:
        ow.set_tolerance(tol, max_sweeps, every)
    t0 = time.perf_counter()
    steps, sweeps = 0, 0
    while True:
        st = ow.step(DT, iters)
        steps += 1
        sweeps += st.iterations
        el = time.perf_counter() - t0
        if el >= budget_s or steps >= 400:
            break
    ow.close()
    return state.n * steps / el, steps, el, sweeps / steps


def cpu_baseline(desc, state, tol, max_sweeps, every, iters, budget_s):
    """The CPU oracle (C++, the same algorithms and sweep rule) continuing from the GPU's state: one
    thread and every host core of this process (at most 16, the box's CPU share)."""
    model, nproc = host_cpu()
    cores = max(1, min(nproc, 16))
    r1, s1, t1, sw1 = oracle_rate(desc, state, tol, max_sweeps, every, iters, 1, budget_s)
    rn, sn, tn, swn = oracle_rate(desc, state, tol, max_sweeps, every, iters, cores, budget_s)
    what = "residual <= %g" % tol if tol > 0 else "%d sweeps" % iters
    return {
        "value": round(rn, 1), "unit": "body-steps/s", "cores": cores, "kind": "port",
        "sample": "oracle (C++ restatement, %d threads) continuing from the GPU state after the timed region, "
                  "%s: %d bodies x %d steps in %.1f s (mean %.1f sweeps)" % (cores, what, state.n, sn, tn, swn),
        "one_thread": {"value": round(r1, 1), "steps": s1, "seconds": round(t1, 2), "mean_sweeps": round(sw1, 2)},
        "cpu_model": model, "nproc": nproc,
    }


def state_of(w, bodies):
    g = w.get_bodies()
    s = bodies.copy()
    s.pos, s.quat, s.lin_vel, s.ang_vel = g.pos, g.quat, g.lin_vel, g.ang_vel
    return s


def kinetic_energy(b, v, w):
    """Translational + rotational kinetic energy (J, FP64) of the dynamic bodies."""
    dyn = b.inv_mass > 0
    m = 1.0 / b.inv_mass[dyn].astype(np.float64)
    ke = 0.5 * (m * (v[dyn].astype(np.float64) ** 2).sum(1)).sum()
    q = b.quat[dyn].astype(np.float64)
    x, y, z, s = q[:, 0], q[:, 1], q[:, 2], q[:, 3]
    R = np.stack([np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - s * z), 2 * (x * z + s * y)], -1),
                  np.stack([2 * (x * y + s * z), 1 - 2 * (x * x + z * z), 2 * (y * z - s * x)], -1),
                  np.stack([2 * (x * z - s * y), 2 * (y * z + s * x), 1 - 2 * (x * x + y * y)], -1)], -2)
    wl = np.einsum("nji,nj->ni", R, w[dyn].astype(np.float64))
    inertia = 1.0 / b.inv_inertia[dyn].astype(np.float64)
    return ke + 0.5 * (inertia * wl * wl).sum()


def fp64_resolve(w, bodies, desc):
    """One more GPU step (FP32) and the FP64 oracle solving the same manifolds from the same state,
    warm start, friction bounds and colours at the same sweep count: the relative difference of the kinetic energy
    after the step (the energy drift of one step against the FP64 re-solve), the largest velocity
    difference, and the FP64 solve's residual."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import orc

    before = state_of(w, bodies)
    st = w.step(DT, max(desc.max_iterations, 1), axm.STEP_RESIDUAL | axm.STEP_KEEP_STAGES)
    man = w.manifolds()
    col, _, _ = w.colours()
    warm, _ = w.impulses()
    bounds = w.friction_bounds()
    after = w.get_bodies()
    d64 = axm.WorldDesc.from_buffer_copy(desc)
    d64.residual_tol = 0.0
    ow = orc.OracleWorld(orc.params_from_desc(d64), fp64=True)
    ow.set_bodies(before)
    ost = ow.step_given(DT, st.iterations, man, warm=warm, colours=col, bounds=bounds)
    _, _, v64, w64 = ow.get_state()
    ow.close()
    e32 = kinetic_energy(bodies, after.lin_vel, after.ang_vel)
    e64 = kinetic_energy(bodies, v64, w64)
    dv = np.abs(after.lin_vel.astype(np.float64) - v64).max()
    return {"sweeps": int(st.iterations), "manifolds": int(st.manifolds), "ke_fp32": e32, "ke_fp64": e64,
            "energy_drift": (e32 - e64) / e64 if e64 else 0.0, "max_dv": float(dv),
            "residual_fp32": float(st.residual), "residual_fp64": float(ost.residual)}


def committed_traffic(kernel, cfg, n, args):
    """HBM bytes per launch of `kernel` from the committed counter runs (FETCH_SIZE and WRITE_SIZE,
    each scaled by what it reads for a plain copy of known size), when they were taken on this
    exact workload; None otherwise."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles",
                        "%s_scene%d_traffic.json" % (kernel.split(" ")[0], cfg))
    try:
        with open(path) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    want = {"config": cfg, "bodies": n, "steps": args.steps, "warmup": args.warmup, "residual_tol": args.tol,
            "max_sweeps": args.max_iters, "check_every": max(1, args.tol_every)}
    if t.get("kernel") != kernel or t.get("workload") != want:
        return None
    return {"bytes_per_launch": t["bytes_per_launch"], "source": "profiles/" + os.path.basename(path)}


def sweep_launches(tot, prof):
    """(bytes, seconds, launches) of the two launches the sweeps are timed in, 240 B per contact point
    and sweep each: the islands each solved by a workgroup or a wave (their points x the sweeps each
    ran), and the rest: the large islands, and those of 257 to 4096 manifolds that the large islands'
    sweep takes along."""
    kern = {"k_pgs_solve (large islands)": (B_SWEEP * float(tot.contact_sweeps - prof.bundle_point_sweeps),
                                            prof.pgs_ms * 1e-3, int(prof.pgs_launches))}
    if prof.bundle_launches:
        kern["k_pgs_solve (other islands)"] = (B_SWEEP * float(prof.bundle_point_sweeps), prof.bundle_ms * 1e-3,
                                               int(prof.bundle_launches))
    return kern


def headline(args):
    cfg = args.config
    bodies, desc = axm.scene(cfg, SEED_BASE + 1000 * cfg, args.bodies, args.worlds)
    iters = args.iters or DEFAULT_ITERS[cfg]
    if args.tol > 0:
        desc.residual_tol = args.tol
        desc.max_iterations = args.max_iters
        desc.residual_every = max(1, args.tol_every)
    log("scene config %d: %d bodies" % (cfg, bodies.n))
    w = axm.World(desc)
    w.set_bodies(bodies)
    sweeps_arg = args.max_iters if args.tol > 0 else iters
    t0 = time.time()
    w.run(DT, sweeps_arg, args.warmup, graph=not args.eager)
    w.sync()
    log("warm-up %d steps (%.1fs)" % (args.warmup, time.time() - t0))
    tuned = None
    if args.autotune and args.tol <= 0:
        # tuned on a copy of the warmed-up state, so the timed world's trajectory is untouched
        tw = axm.World(desc)
        tw.set_bodies(state_of(w, bodies))
        tw.step(DT, iters, 0)
        g, lds, pol, ms = tw.autotune(DT, iters, 5)
        tw.close()
        w.set_sweep_config(g, lds, pol)
        tuned = {"groups": g, "lds_kib": lds, "policy": pol, "sweep_ms": round(ms, 4)}
    # The timed steps run `repeats` times from the same warmed-up state (a snapshot of the world,
    # reloaded before each run; the run with the median time is reported).  Two untimed profiled
    # steps first capture the profiled step graphs of both warm-start parities, which the reload
    # keeps, so no run pays for a capture.
    snap = os.path.join(tempfile.gettempdir(), "axm_bench_%d.snapshot" % os.getpid())
    w.save(snap)
    w.profile(True)
    w.run(DT, sweeps_arg, 2, graph=not args.eager)
    w.profile(False)
    runs = []
    try:
        for rep in range(max(1, args.repeats)):
            w.load(snap)
            w.totals(reset=True)
            w.profile(True)
            w.sync()
            t0 = time.perf_counter()
            w.run(DT, sweeps_arg, args.steps, graph=not args.eager)
            w.sync()
            el = time.perf_counter() - t0
            runs.append((el, w.profile(False), w.totals(reset=True)))
    finally:
        os.remove(snap)
    order = sorted(range(len(runs)), key=lambda i: runs[i][0])
    elapsed, prof, tot = runs[order[len(order) // 2]]
    log("timed %d steps %d times: median %.4fs (min %.4fs, max %.4fs)" % (
        args.steps, len(runs), elapsed, runs[order[0]][0], runs[order[-1]][0]))
    diag = w.step(DT, sweeps_arg, axm.STEP_RESIDUAL | axm.STEP_TIMINGS)
    value = bodies.n * args.steps / elapsed
    steps_done = max(int(tot.steps), 1)
    mean_sweeps = tot.sweeps / steps_done
    kern = sweep_launches(tot, prof)  # the roofline line is the one with more time

    def roof_of(name):
        nbytes, secs, n = kern[name]
        n = max(n, 1)
        ach = nbytes / secs / 1e9 if secs > 0 else 0.0
        return {
            "bound": "hbm", "achieved": round(ach, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(ach / HBM_PEAK_GBS, 5), "traffic": None, "kernel": name,
            "launches": int(kern[name][2]), "avg_launch_us": round(secs * 1e6 / n, 3),
            "bytes_per_launch": round(nbytes / n, 1),
            "per_unit": "240 B per contact point per sweep", "share_of_step": round(secs / elapsed, 4),
        }
    dominant = max(kern, key=lambda k: kern[k][1])
    roof = roof_of(dominant)
    traffic = committed_traffic(dominant, cfg, bodies.n, args)
    if traffic:
        roof["traffic"] = traffic["bytes_per_launch"]
        roof["traffic_source"] = traffic["source"]
    # whole step: 304 N + 104 P + 304 C + 12 R C + 240 I C per step (P, C, R of the diagnostic step)
    dyn = int((bodies.inv_mass > 0).sum())
    b_step = (B_BODY * dyn + B_PAIR * diag.pairs + B_CONTACT * diag.contacts + B_ROUND * diag.colour_rounds *
              diag.contacts) + B_SWEEP * float(tot.contact_sweeps) / steps_done
    step_gbs = b_step * args.steps / elapsed / 1e9
    out = {
        "metric": "body-steps/sec at contact residual <=1e-4: plain GPU vs batched+learned warm-start",
        "value": round(value, 1),
        "unit": "body-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(elapsed * 1e3 / args.steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded DeterministicRNG scene)",
        "config": {
            "workload": WORKLOADS[cfg], "scene_config": cfg, "bodies": bodies.n, "dt": DT,
            "residual_tol": args.tol, "max_sweeps": sweeps_arg if args.tol > 0 else None,
            "residual_check_every": max(1, args.tol_every) if args.tol > 0 else None,
            "sweeps": None if args.tol > 0 else iters, "softness": round(float(desc.softness), 4),
            "mode": "plain GPU, previous-step warm start" + (", residual-stopped" if args.tol > 0 else ""),
            "launch": "eager" if args.eager else "hipGraph replay",
            "sweep_launch": tuned if tuned else "default (one workgroup per CU)",
        },
        "at_tolerance": {
            "steps": int(tot.steps), "steps_at_tol": int(tot.steps_at_tol),
            "fraction_reached": round(tot.steps_at_tol / steps_done, 4) if args.tol > 0 else None,
            "mean_sweeps": round(mean_sweeps, 2), "max_sweeps_used": int(tot.max_sweeps),
            "contact_point_sweeps_per_step": round(tot.contact_sweeps / steps_done, 1),
            "island_share_of_point_sweeps": round(tot.local_contact_sweeps / max(tot.contact_sweeps, 1), 4),
        },
        "last_step": {k: diag.as_dict()[k] for k in ("pairs", "manifolds", "contacts", "colours", "colour_rounds",
                                                    "iterations", "residual", "broadphase_ms", "narrowphase_ms",
                                                    "solver_ms", "integration_ms", "total_ms")},
        "timing": {"repeats": len(runs), "from": "the same warmed-up state (snapshot reloaded)",
                   "seconds": [round(r[0], 5) for r in runs], "reported": "median"},
        "roofline": roof,
        "roofline_sweep_kernels": {k: roof_of(k) for k in kern},
        "roofline_step": {"bytes_per_step": round(b_step, 1), "achieved": round(step_gbs, 2), "unit": "GB/s",
                          "frac": round(step_gbs / HBM_PEAK_GBS, 5),
                          "formula": "304 N + 104 P + 304 C + 12 R C + 240 I C"},
    }
    if not args.no_fp64:
        r = fp64_resolve(w, bodies, desc)
        out["fp64_resolve"] = {k: (float("%.6g" % v) if isinstance(v, float) else v) for k, v in r.items()}
        log("fp64 re-solve: energy drift %.3g, max dv %.3g" % (r["energy_drift"], r["max_dv"]))
    state = state_of(w, bodies) if not args.no_cpu else None
    w.close()
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(desc, state, args.tol, args.max_iters, max(1, args.tol_every), iters,
                                           args.cpu_seconds)
        out["gpu_over_cpu"] = round(value / out["cpu_baseline"]["value"], 2)
        out["gpu_over_cpu_1thread"] = round(value / out["cpu_baseline"]["one_thread"]["value"], 2)
    return out


def pile_section(steps, no_cpu, cpu_seconds):
    """The dense pile (100k bodies, 20 sweeps) over the configuration's full run of `steps` steps from
    its initial state: body-steps/s, contacts at the end, the sweep kernel's share."""
    bodies, desc = axm.scene(1, SEED_BASE + 1000, 0, 0)
    w = axm.World(desc)
    w.set_bodies(bodies)
    w.step(DT, 20, 0)
    w.sync()
    w.totals(reset=True)
    t0 = time.perf_counter()
    w.run(DT, 20, steps - 1, graph=True)
    w.sync()
    el = time.perf_counter() - t0
    tot = w.totals(reset=True)
    diag = w.step(DT, 20, axm.STEP_RESIDUAL)
    out = {"workload": WORKLOADS[1], "bodies": bodies.n, "sweeps": 20, "steps": steps - 1,
           "body_steps_per_s": round(bodies.n * (steps - 1) / el, 1), "ms_per_step": round(el * 1e3 / (steps - 1), 4),
           "contacts_last_step": int(diag.contacts), "manifolds_last_step": int(diag.manifolds),
           "contacts_per_body": round(diag.contacts / bodies.n, 3), "colours": int(diag.colours),
           "mean_contacts": round(tot.contact_sweeps / max(tot.sweeps, 1), 1),
           "residual_last_step": float(diag.residual)}
    log("pile: %.0f body-steps/s, %d contacts at the end" % (out["body_steps_per_s"], diag.contacts))
    if not no_cpu:
        out["cpu_baseline"] = cpu_baseline(desc, state_of(w, bodies), 0.0, 0, 1, 20, cpu_seconds)
    w.close()
    return out


def settled(cfg, seed, n, worlds, steps, sweeps):
    """The state of a scene after `steps` plain steps at a fixed sweep count (graph replay)."""
    b, d = axm.scene(cfg, seed, n, worlds)
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, sweeps, steps, graph=True)
    s = state_of(w, b)
    w.close()
    return s, d


def tolerance_comparison(tol, max_sweeps, worlds):
    """Body-steps/s and sweeps per step when every step iterates to residual <= tol: the plain
    previous-step warm start against the learned one (network trained here on the GPU on contacts
    logged from the plain solver on seeded dense piles), on a held-out dense pile settled for 300
    steps and on a batch of `worlds` independent worlds after 60 steps."""
    import warmstart

    t0 = time.time()
    net, losses, rows = warmstart.train_default()
    out = {"residual_tol": tol, "max_sweeps": max_sweeps,
           "training": {"rows": rows, "epochs": len(losses), "loss_first": round(float(losses[0]), 5),
                        "loss_last": round(float(losses[-1]), 5), "seconds": round(time.time() - t0, 2),
                        "data": warmstart.TRAIN_DATA}}
    log("warm-start network trained on %d contacts in %.1fs" % (rows, time.time() - t0))
    pile, dp = settled(1, SEED_BASE + 1000 + 2 * 200, 0, 0, 300, 20)
    batch, db = settled(3, SEED_BASE + 3000, 0, worlds, 60, 10)
    cases = (("pile_plain", pile, dp, axm.WARM_CACHE, None, 3, 20),
             ("pile_learned", pile, dp, axm.WARM_MLP, net, 3, 20),
             ("batched_plain", batch, db, axm.WARM_CACHE, None, 3, 30),
             ("batched_learned", batch, db, axm.WARM_MLP, net, 3, 30))
    for name, bb, dd, warm, nn, warmup, steps in cases:
        tm = {}
        it, reached = warmstart.iterations_to_tolerance(bb, dd, steps, tol, max_sweeps, warm, net=nn, warmup=warmup,
                                                        every=1, timing=tm)
        out[name] = {"bodies": bb.n, "steps": steps, "body_steps_per_s": round(bb.n * steps / tm["s"], 1),
                     "mean_sweeps": round(float(it.mean()), 2), "median_sweeps": float(np.median(it)),
                     "fraction_reached": round(float(reached.mean()), 3)}
        log("%s: %.0f body-steps/s, mean sweeps %.1f, reached %.2f" % (name, out[name]["body_steps_per_s"],
                                                                       it.mean(), reached.mean()))
    for kind in ("pile", "batched"):
        p, l_ = out[kind + "_plain"], out[kind + "_learned"]
        out[kind + "_gain"] = {"sweeps_ratio": round(p["mean_sweeps"] / max(l_["mean_sweeps"], 1e-9), 3),
                               "rate_ratio": round(l_["body_steps_per_s"] / max(p["body_steps_per_s"], 1e-9), 3)}
    net.close()
    return out


def mlp_forward_rate(rows, reps):
    """Inference of the warm-start network on `rows` synthetic contact points, `reps` times
    (the rocprof kernel time of k_mlp_forward gives the MFMA rate: 2 x (32x128 + 128x128 +
    128x16) FLOP per row at the padded MFMA shapes, 2 x (24x128 + 128x128 + 128x3) useful)."""
    rng = np.random.default_rng(5)
    X = rng.normal(size=(rows, axm.MLP_INPUTS)).astype(np.float32)
    net = axm.Mlp(0, seed=3)
    t0 = time.perf_counter()
    for _ in range(reps):
        net.forward(X)
    el = time.perf_counter() - t0
    net.close()
    print(json.dumps({"mlp_forward": {"rows": rows, "reps": reps, "seconds_with_copies": round(el, 4),
                                      "flop_per_row_padded": 2 * (32 * 128 + 128 * 128 + 128 * 16),
                                      "flop_per_row_useful": 2 * (24 * 128 + 128 * 128 + 128 * 3)}}), flush=True)


def copy_calibration(mib, reps):
    """Plain device-to-device copies of a known size (read `mib` MiB, write `mib` MiB per
    dispatch), for scaling the HBM counters FETCH_SIZE / WRITE_SIZE of a counter run.
    Uses PyTorch only (the physics library is not loaded in this mode)."""
    import torch

    n = mib * (1 << 20) // 4
    a = torch.ones(n, dtype=torch.float32, device="cuda:0")
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    for _ in range(reps):
        b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration": {"bytes_read": n * 4, "bytes_written": n * 4, "dispatches": reps}}),
          flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=110)
    ap.add_argument("--repeats", type=int, default=5, help="timed runs from the same state (median reported)")
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--config", type=int, default=2)
    ap.add_argument("--bodies", type=int, default=0)
    ap.add_argument("--worlds", type=int, default=0)
    ap.add_argument("--iters", type=int, default=0, help="fixed sweeps per step (with --tol 0)")
    ap.add_argument("--tol", type=float, default=1e-4, help="iterate each step until the residual <= tol (0: fixed)")
    ap.add_argument("--max-iters", type=int, default=300)
    ap.add_argument("--tol-every", type=int, default=1, help="with --tol: sweeps between residual checks")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fp64", action="store_true", help="skip the FP64 re-solve of one step")
    ap.add_argument("--eager", action="store_true", help="launch every step's kernels instead of replaying a graph")
    ap.add_argument("--autotune", action="store_true", help="autotune the sweep launch shape (fixed sweeps only)")
    ap.add_argument("--no-pile", action="store_true", help="skip the dense pile section")
    ap.add_argument("--pile-steps", type=int, default=600)
    ap.add_argument("--no-tolerance", action="store_true", help="skip the plain vs learned run at residual <= tol")
    ap.add_argument("--tolerance-worlds", type=int, default=4096)
    ap.add_argument("--mlp-forward", type=int, default=0, metavar="ROWS",
                    help="only run the warm-start network's inference on ROWS synthetic rows (MFMA rate)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="only run plain copies of MIB MiB (counter scaling), then exit")
    args = ap.parse_args()
    if args.copy_calibration:
        copy_calibration(args.copy_calibration, 5)
        return
    if args.mlp_forward:
        mlp_forward_rate(args.mlp_forward, 5)
        return
    if args.gpus != 1:
        print("bench.py measures one GPU: this build is single-GPU (every box has one MI355X); "
              "--gpus %d is not supported" % args.gpus, file=sys.stderr)
        sys.exit(2)
    if axm.device_count() < 1:
        print("no HIP device visible", file=sys.stderr)
        sys.exit(1)
    out = headline(args)
    if not args.no_pile:
        out["pile_100k"] = pile_section(args.pile_steps, args.no_cpu, args.cpu_seconds)
    if not args.no_tolerance:
        out["plain_vs_learned"] = tolerance_comparison(1e-4, args.max_iters, args.tolerance_worlds)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
