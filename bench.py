"""Benchmark of the DNS + droplet time step on one MI355X.

Workload (the configuration the headline metric is quoted on): 256^3 periodic box,
deterministic forcing, 1,000,000 droplets with log-normal radii (median 25 um,
sigma_ln 0.4, clipped to 5-60 um), hydrodynamic interactions with a cutoff of 50
radii, collision detection and statistics.  A "step" is one full time step of the
flow and of every droplet.  Synthetic inputs: seeded initial flow and droplets,
generated before the timed region; all state is resident in HBM.

Prints ONE JSON line.  value = FP32-mixed steps/s; the FP64 path is timed on the same
workload for the speed-up.  Accuracy is stated against the FP64 oracle (the project's
CPU restatement of the reference algorithm): the velocity relative L2 and the per-shell
E(k) error after 10 steps, and the collision kernel and contact RDF of the FP32-mixed
path next to the oracle's over the steps of the CPU baseline, with Poisson error bars.
The CPU baseline times the oracle on a bounded sample of the same workload.
"""
from __future__ import annotations

import argparse
import functools
import json
import os
import statistics
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import mpi_2d_domain_decomp_turb_particles_amd as dd  # noqa: E402

HBM_PEAK_GBS = 8000.0
WORKLOAD = "256^3 DNS (deterministic forcing) + 1M log-normal droplets, HI 50 radii, collisions"
FFT_KERNELS = ("y_inv", "x_fused", "y_fwd", "z_stage")


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def workload_params(precision: int, N: int = 256, npart: int = 1_000_000):
    # parameter.d_256_det: rnu 0.002, dt 0.001, eta/tau_K 0.01392/0.09694, force 1.242477/0.391356
    return dd.default_params(
        N=N, precision=precision, dt=0.001, rnu=0.002, forcing=1, force=(1.242477, 0.391356),
        etk_DNS=0.01392, tauk_DNS=0.09694, npart=npart, nset=10,
        radius=[5.0, 10.0, 15.0, 20.0, 25.0, 30.0, 35.0, 40.0, 50.0, 60.0],
        hdi_included=1, hdi_trunc=50.0, nonoverlap=1,
    )


def make_solver(precision, N, npart, seed_flow=123, seed_drop=290710):
    s = dd.Solver(workload_params(precision, N, npart))
    s.init_flow(dd.SPEC_K4_GAUSS, seed_flow, 4.0, 1.0)
    s.init_droplets(seed=seed_drop, radii=dd.RADII_LOGNORMAL, median_um=25.0, sigma_ln=0.4, rmin_um=5.0, rmax_um=60.0)
    return s


def solver_from(state, precision, N, npart):
    s = dd.Solver(workload_params(precision, N, npart))
    s.set_flow(*state["flow"])
    d = state["drop"]
    s.set_droplets(d["yp"], d["fvp"], d["fdp"], d["pertvel"])
    return s


@functools.lru_cache(maxsize=None)
def sphere_fraction(N: int) -> float:
    """Fraction of the stored modes (kx < N/2, all ky, kz) inside the dealiasing sphere:
    shell int(|k| + 1/2) <= nek = N/2 - 1.5, the mean mode counted inside.  Beyond it the
    state and the stored nonlinear term are zero, and the z stage neither reads nor writes
    them once a step has."""
    nek = int(N / 2 - 1.5)
    w = np.arange(N)
    w = np.where(w <= N // 2, w, w - N).astype(np.float64)
    r2 = (w[:, None] ** 2 + w[None, :] ** 2)
    inside = 0
    for kx in range(N // 2):
        k2 = r2 + kx * kx
        if kx == 0:
            k2 = k2.copy()
            k2[0, 0] = 1e-5
        inside += int(np.count_nonzero(np.floor(np.sqrt(k2) + 0.5) <= nek))
    return inside / (N * N * (N // 2))


def column_fraction(N: int) -> float:
    """Fraction of the (kx, ky) columns with a mode inside the dealiasing sphere."""
    nek = int(N / 2 - 1.5)
    k = np.arange(N)
    k = np.where(k > N // 2, k - N, k)
    k2 = np.arange(N // 2)[:, None] ** 2 + (k ** 2)[None, :]
    return float((k2 <= nek * (nek + 1)).mean())


def kernel_bytes(N: int, prec: int):
    """Compulsory HBM bytes per launch of each flow kernel (every input read once,
    every output written once).  C = one complex field N*N*(N/2), R = one real field."""
    cs = 16 if prec == dd.FP64 else 8
    rs = cs // 2
    C = N * N * (N // 2) * cs
    R = N * N * N * rs
    f, g = sphere_fraction(N), column_fraction(N)
    return {
        "y_inv": int(6 * g * C) + 6 * C,    # 6 fields, read inside the sphere's columns only
        "x_fused": 6 * C + 3 * C + 3 * R,   # read u, w; write u x w and the physical u
        "y_fwd": 3 * C + int(3 * g * C),
        "pre": 0,
        # one kernel at every N: reads N (3C) and writes the six inverse outputs (6C) in the
        # sphere's columns, reads and writes u, o (12C) inside the sphere
        "z_stage": int((9 * g + 12 * f) * C),
        "sym": 0,
    }


def measured_traffic(kernel, N, prec):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 --pmc summary
    (FETCH_SIZE + WRITE_SIZE, scaled by the copy-kernel calibration), or None."""
    path = os.path.join(ROOT, "profiles", "hbm_traffic.json")
    try:
        with open(path) as f:
            tab = json.load(f)
    except (OSError, ValueError):
        return None
    key = f"{kernel}/N{N}/{'fp64' if prec == dd.FP64 else 'fp32'}"
    ent = tab.get(key)
    return None if ent is None else ent.get("bytes_per_launch")


def timed_run(s, steps, warmup):
    if warmup:
        s.step(warmup)
    t0 = time.perf_counter()
    st = s.step(steps)
    t1 = time.perf_counter()
    return (t1 - t0), s.timing(), st


def rel_l2(a, b):
    num = sum(float(np.sum((x - y) ** 2)) for x, y in zip(a, b))
    den = sum(float(np.sum(y ** 2)) for y in b)
    return (num / den) ** 0.5


def accuracy_vs_oracle(N, npart, state, steps=10):
    """The FP32-mixed and FP64 GPU paths (with their droplets) and the oracle's flow
    (which does not see the droplets) run `steps` steps from the same state."""
    from oracle import oracle as O
    out = {}
    vel = {}
    spec = {}
    for prec, name in ((dd.FP32_MIXED, "fp32_mixed"), (dd.FP64, "fp64")):
        with solver_from(state, prec, N, npart) as s:
            s.step(steps)
            vel[name] = s.get_flow()[0]
            spec[name] = s.spectrum()
    with O.Oracle(workload_params(dd.FP64, N, 0)) as o:
        o.set_flow(*state["flow"])
        o.flow_only(True)
        o.step(steps)
        vo = o.get_flow()[0]
        eo = o.spectrum()
    live = eo > 1e-12 * eo.max()
    for name in ("fp32_mixed", "fp64"):
        out[f"vel_rel_l2_{steps}_steps_{name}_vs_oracle"] = rel_l2(vel[name], vo)
        out[f"ek_shell_max_rel_err_{name}_vs_oracle"] = float(np.max(np.abs(spec[name][live] / eo[live] - 1)))
    out["vel_rel_l2_10_steps_fp32_vs_fp64"] = rel_l2(vel["fp32_mixed"], vel["fp64"])
    out["ek_shells_compared"] = int(live.sum())
    return out


def contact_pairs_uniform(radii, st_percent, volume):
    """Expected number of droplet pairs with R < d <= R (1 + st/100), R = a_i + a_j,
    for uniformly random positions: sum over i < j of the shell volume over the box
    volume.  With S_k = sum a^k, sum_{i<j} (a_i + a_j)^3 = n S3 + 3 S1 S2 - 4 S3."""
    a = np.asarray(radii, dtype=np.float64)
    n = a.size
    s1, s2, s3 = a.sum(), (a ** 2).sum(), (a ** 3).sum()
    pair_r3 = n * s3 + 3 * s1 * s2 - 4 * s3
    return 4.0 * np.pi / 3.0 * ((1 + st_percent / 100.0) ** 3 - 1) * pair_r3 / volume


def cpu_baseline_and_statistics(N, npart, state, steps):
    """The FP64 oracle on the same workload: one untimed step (the droplet history
    start), then `steps` timed steps; the FP32-mixed GPU path runs the same steps from
    the same state.  Returns the CPU rate and the collision kernel / contact RDF of
    both, summed over all the steps, with Poisson (counting) error bars."""
    from oracle import oracle as O
    p = workload_params(dd.FP64, N, npart)
    o = O.Oracle(p)
    o.set_flow(*state["flow"])
    d = state["drop"]
    o.set_droplets(d["yp"], d["fvp"], d["fdp"], d["pertvel"])
    o.set_new_particle(1)
    g = solver_from(state, dd.FP32_MIXED, N, npart)
    tot = {"oracle": np.zeros(3), "gpu": np.zeros(3)}          # collisions, contacts, pairs within 10 R
    secs = []
    for k in range(1 + steps):
        t0 = time.perf_counter()
        o.step(1)
        dt = time.perf_counter() - t0
        if k > 0:
            secs.append(dt)
        g.step(1)
        for name, x in (("oracle", o), ("gpu", g)):
            c = x.collision_counts()
            tot[name] += (sum(c.icc), sum(c.nir), c.pairs_in_dstat)
        log(f"CPU baseline step {k + 1}/{1 + steps}: {dt:.1f} s")
    threads = O.lib().orc_num_threads()
    o.close()
    g.close()
    nsteps = 1 + steps
    dtime = p.dt
    volume = (2 * np.pi) ** 3
    expect = contact_pairs_uniform(state["drop"]["yp"][6], p.st, volume)

    def stat(name, k):
        v = float(tot[name][k])
        return {"count": v, "sigma": v ** 0.5}

    stats = {
        "steps": nsteps,
        "collision_kernel": {
            "unit": "collisions per unit time per unit volume (DNS units)",
            **{name: {"value": tot[name][0] / (nsteps * dtime * volume),
                      "sigma": tot[name][0] ** 0.5 / (nsteps * dtime * volume),
                      "collisions": int(tot[name][0])} for name in ("gpu", "oracle")},
        },
        "rdf_at_contact": {
            "unit": "contact pairs / expected for uniform positions (R < d <= R(1+st%))",
            **{name: {"value": tot[name][1] / (nsteps * expect),
                      "sigma": tot[name][1] ** 0.5 / (nsteps * expect),
                      "contacts": int(tot[name][1])} for name in ("gpu", "oracle")},
        },
        "pairs_within_10R": {name: stat(name, 2) for name in ("gpu", "oracle")},
        "gpu": "fp32-mixed", "oracle": "fp64",
    }
    return 1.0 / statistics.median(secs), statistics.median(secs), threads, stats


def coalescence_1024(steps, warmup):
    """The 1024^3 configuration: FP32-mixed, stochastic forcing, 5,000,000 droplets of
    15 um growing by coalescence from the first step, HI to 50 radii, collisions.  nu for
    k_max eta ~ 1.5 (eta ~ 4.8e-3, tau_K ~ 0.028 at u' ~ 1), dt at CFL ~ 0.1.  Reported
    beside the headline, not as it: steps/s and the flow kernels' HBM rates."""
    p = dd.default_params(N=1024, precision=dd.FP32_MIXED, dt=0.00025, rnu=0.0008, forcing=2,
                          etk_DNS=0.00476, tauk_DNS=0.0283, npart=5_000_000, nset=1, radius=[15.0],
                          hdi_included=1, hdi_trunc=50.0, nonoverlap=1, nstep_grow=1)
    log("set-up 1024^3, 5M droplets")
    with dd.Solver(p) as s:
        t0 = time.perf_counter()
        s.init_flow(dd.SPEC_K4_GAUSS, 123, 4.0, 1.0)
        s.init_droplets(seed=290710)
        setup = time.perf_counter() - t0
        el, t, _ = timed_run(s, steps, warmup)
        n = s.get_droplets()["yp"].shape[1]
        alone = s.profile_flow(2)
        tune = s.tuning()
        copy_ms, copy_bytes = s.profile_copy(5)
    kb = kernel_bytes(1024, dd.FP32_MIXED)
    kms = dict(zip(["y_inv", "x_fused", "y_fwd", "pre", "z_stage", "sym"], t.flow_kernel_ms))
    return {
        "workload": "1024^3 DNS (stochastic forcing) + 5M droplets of 15 um, coalescence from step 1, HI 50 radii",
        "steps": steps, "warmup": warmup, "steps_per_s": steps / el, "ms_per_step": 1e3 * el / steps,
        "setup_s": setup, "droplets_after": n,
        "phase_ms_per_step": {"flow": t.flow_ms / steps, "cells": t.cells_ms / steps, "interp": t.interp_ms / steps,
                              "hdi": t.hdi_ms / steps, "advance": t.advance_ms / steps,
                              "colldet": t.colldet_ms / steps, "overlap": t.overlap_ms / steps},
        "flow_kernels_GBps_in_step": {k: kb[k] / (kms[k] / steps * 1e-3) / 1e9 for k in FFT_KERNELS if kms[k] > 0},
        "flow_kernels_GBps_alone": {k: kb[k] / (alone[k] * 1e-3) / 1e9 for k in FFT_KERNELS if alone[k] > 0},
        "tuning": {k: (v.tolist() if hasattr(v, "tolist") else v) for k, v in tune.items()},
        "hbm_copy_GBps": copy_bytes / (copy_ms * 1e-3) / 1e9,
    }


def batched_48x64(steps, warmup, R=48, N=64, compare=True):
    """The batched configuration: 48 independent 64^3 realisations (different seeds,
    deterministic and stochastic forcing alternating), FP32-mixed, droplet counts drawn
    uniformly from 5,000-200,000 per realisation, one droplet size per realisation with
    Stokes numbers 0.2-3, HI (truncation at 50 radii or fewer, about 24 neighbours per
    droplet on average), collisions and relocation.  All realisations advance in one
    ddns_batch_step: every flow stage is one launch over the 48 fields, replayed from HIP
    graphs, and the droplet blocks run beside it.  The same realisations stepped one
    handle after another are timed for comparison."""
    params = dd.batched_realisations(R=R, N=N, precision=dd.FP32_MIXED)
    ndrop = sum(p.npart for p in params)
    log(f"set-up {R} x {N}^3, {ndrop} droplets")
    t0 = time.perf_counter()
    with dd.Batch(params) as b:
        for r, p in enumerate(params):
            m = b.member(r)
            m.init_flow(dd.SPEC_K4_GAUSS, p.iseed_m0, 4.0, 1.0)
            m.init_droplets(seed=290710 + r)
        setup = time.perf_counter() - t0
        if warmup:
            b.step(warmup)
        t1 = time.perf_counter()
        b.step(steps)
        el = time.perf_counter() - t1
        t = b.timing()
        tune = b.tuning()
        iters = [b.member(r).collision_counts().gmres_iters for r in range(R)]
    log(f"batched: {1e3 * el / steps:.2f} ms per step")
    seq_steps = max(2, steps // 4)
    seq = 0.0
    for r, p in enumerate(params if compare else []):
        with dd.Solver(p) as s:
            s.init_flow(dd.SPEC_K4_GAUSS, p.iseed_m0, 4.0, 1.0)
            s.init_droplets(seed=290710 + r)
            s.step(1)
            t2 = time.perf_counter()
            s.step(seq_steps)
            seq += time.perf_counter() - t2
    seq_ms = 1e3 * seq / seq_steps if compare else None
    ms = 1e3 * el / steps
    return {
        "metric": "realisation-steps/s, 48 x 64^3 realisations with 5k-200k droplets each, FP32-mixed, one GPU",
        "value": R * steps / el, "unit": "realisation-steps/s", "higher_is_better": True,
        "n_gpus": 1, "steps": steps, "warmup": warmup, "ms_per_step": ms, "dtype": "fp32-mixed",
        "data": "synthetic (random-phase initial fields, uniform droplet positions)",
        "config": {"workload": f"{R} x {N}^3 DNS + {ndrop} droplets in total (5k-200k per realisation), St 0.2-3, "
                               "mixed deterministic/stochastic forcing, HI, collisions", "realisations": R, "N": N,
                   "droplets": ndrop, "parallelism": "single GPU"},
        "droplet_updates_per_s": ndrop * steps / el,
        "setup_s": setup,
        "flow_ms_per_step": t.flow_ms / steps,
        "droplet_phase_ms_per_step_summed_over_realisations": {
            "cells": t.cells_ms / steps, "interp": t.interp_ms / steps, "hdi": t.hdi_ms / steps,
            "advance": t.advance_ms / steps, "colldet": t.colldet_ms / steps, "overlap": t.overlap_ms / steps},
        "gmres_iterations": {"min": min(iters), "max": max(iters)},
        "separate_handles_ms_per_step": seq_ms,
        "speedup_vs_separate_handles": seq_ms / ms if compare else None,
        "tuning": {k: (v.tolist() if hasattr(v, "tolist") else v) for k, v in tune.items()},
    }


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--N", type=int, default=256)
    ap.add_argument("--npart", type=int, default=1_000_000)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-steps", type=int, default=3)
    ap.add_argument("--no-accuracy", action="store_true")
    ap.add_argument("--no-compare", action="store_true",
                    help="batch-48x64: skip the timing of the same realisations as separate handles")
    ap.add_argument("--only-fp32", action="store_true",
                    help="time the FP32-mixed path only (for profiler runs)")
    ap.add_argument("--workload", choices=["headline", "coalescence-1024", "batch-48x64"], default="headline",
                    help="coalescence-1024: the 1024^3 + 5M-droplet configuration instead; batch-48x64: the 48 "
                         "batched 64^3 realisations (one JSON line of its own each)")
    a = ap.parse_args(argv)
    if a.gpus != 1:
        print(f"bench.py measures one GPU: the whole periodic domain lives on a single MI355X; --gpus {a.gpus} is not supported", file=sys.stderr)
        return 2
    if a.workload == "coalescence-1024":
        print(json.dumps(coalescence_1024(a.steps, a.warmup)))
        return 0
    if a.workload == "batch-48x64":
        print(json.dumps(batched_48x64(a.steps, a.warmup, compare=not a.no_compare)))
        return 0
    N, npart = a.N, a.npart

    # ---- FP32-mixed (the value)
    log(f"set-up N={N} droplets={npart}")
    s32 = make_solver(dd.FP32_MIXED, N, npart)
    log("FP32-mixed timed run")
    init_state = {"flow": s32.get_flow(), "drop": s32.get_droplets()}
    el32, t32, st = timed_run(s32, a.steps, a.warmup)
    cc = s32.collision_counts()
    steps_per_s = a.steps / el32
    kms = list(t32.flow_kernel_ms)
    names = ["y_inv", "x_fused", "y_fwd", "pre", "z_stage", "sym"]
    per_launch = {n: kms[i] / a.steps for i, n in enumerate(names)}
    kb = kernel_bytes(N, dd.FP32_MIXED)
    flow_ms = t32.flow_ms / a.steps
    # the flow step alone (no droplet block beside it), after the timed run
    alone = s32.profile_flow(5)
    tune = {k: (v.tolist() if hasattr(v, "tolist") else v) for k, v in s32.tuning().items()}
    copy_ms, copy_bytes = s32.profile_copy(20)
    s32.close()
    # by the times alone: beside the droplet block a launch's time depends on what it meets
    dom = max(FFT_KERNELS, key=lambda n: alone[n])
    achieved = kb[dom] / (per_launch[dom] * 1e-3) / 1e9
    achieved_alone = kb[dom] / (alone[dom] * 1e-3) / 1e9
    flow_kernels = {
        n: {"bytes": kb[n], "ms_in_step": per_launch[n], "ms_alone": alone[n],
            "GBps_in_step": kb[n] / (per_launch[n] * 1e-3) / 1e9, "GBps_alone": kb[n] / (alone[n] * 1e-3) / 1e9}
        for n in FFT_KERNELS
    }
    phases = {"flow": flow_ms, "cells": t32.cells_ms / a.steps, "interp": t32.interp_ms / a.steps,
              "hdi": t32.hdi_ms / a.steps, "advance": t32.advance_ms / a.steps,
              "colldet": t32.colldet_ms / a.steps, "overlap": t32.overlap_ms / a.steps}
    if a.only_fp32:
        print(json.dumps({"metric": "fp32-mixed steps/s (profiling run)", "value": steps_per_s,
                          "ms_per_step": 1e3 * el32 / a.steps, "flow_kernels": flow_kernels,
                          "phase_ms_per_step": phases, "gmres_iters_last_step": cc.gmres_iters}))
        return 0

    # ---- FP64 plain path, same initial state
    log(f"FP32-mixed {steps_per_s:.3f} steps/s; FP64 timed run")
    s64 = solver_from(init_state, dd.FP64, N, npart)
    el64, t64, _ = timed_run(s64, a.steps, a.warmup)
    fp64_sps = a.steps / el64
    s64.close()

    # ---- accuracy against the FP64 oracle after 10 steps
    acc = {}
    if not a.no_accuracy:
        log(f"FP64 {fp64_sps:.3f} steps/s; accuracy run (10 steps, GPU and oracle)")
        try:
            acc = accuracy_vs_oracle(N, npart, init_state)
        except Exception as e:  # reported, never required
            print(f"accuracy run failed: {e}", file=sys.stderr)

    # ---- CPU baseline (oracle, FP64) on a bounded sample, with collision statistics
    cpu, stats = None, None
    if not a.no_cpu:
        log("CPU baseline")
        try:
            sps, med, threads, stats = cpu_baseline_and_statistics(N, npart, init_state, a.cpu_steps)
            cpu = {"value": sps, "unit": "steps/s", "cores": threads, "kind": "port",
                   "sample": f"median of {a.cpu_steps} full steps of the same workload ({med:.1f} s each) after one "
                             f"untimed step, FP64 oracle, {threads} OpenMP threads"}
        except Exception as e:  # the baseline is reported, never required
            print(f"cpu baseline failed: {e}", file=sys.stderr)

    out = {
        "metric": "steps/s at 256^3+1M droplets, FP32-mixed vs FP64 on 1 GPU, vel err <=1e-5",
        "value": steps_per_s,
        "unit": "steps/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": 1e3 * el32 / a.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32-mixed (f32 flow + HI, f64 droplets)",
        "data": "synthetic",
        "config": {"workload": WORKLOAD, "N": N, "droplets": npart, "parallelism": "single GPU"},
        "fp64_steps_per_s": fp64_sps,
        "speedup_fp32_mixed_vs_fp64": steps_per_s / fp64_sps,
        **acc,
        "droplet_updates_per_s": steps_per_s * npart,
        "pairs_tested_per_s": cc.pairs_tested / (t32.colldet_ms / a.steps * 1e-3) if t32.colldet_ms > 0 else None,
        "gmres_iters_last_step": cc.gmres_iters,
        "flow_ms_per_step": flow_ms,
        "flow_ms_per_step_alone": alone["step"],
        "flow_algorithmic_GBps": sum(kb.values()) / (flow_ms * 1e-3) / 1e9,
        "phase_ms_per_step": phases,
        "flow_kernels": flow_kernels,
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": measured_traffic(dom, N, dd.FP32_MIXED),
                     "algorithmic_bytes": kb[dom],
                     "timing": "frac: mean launch time in the last and every 16th of the timed steps "
                               "(HIP events on the flow stream, with the droplet block running beside it); "
                               "frac_alone: the flow step alone",
                     "achieved_alone": achieved_alone, "frac_alone": achieved_alone / HBM_PEAK_GBS},
        "hbm_copy_GBps": copy_bytes / (copy_ms * 1e-3) / 1e9,
        "tuned_shapes": tune,
        "collision_statistics": stats,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out))
    return 0


if __name__ == "__main__":
    raise SystemExit(main())
