"""Benchmark of the force-evaluation path on one MI355X.

Headline (`value`): FP32 split-precision direct sum + Leapfrog.  One "step" =
one Leapfrog KDK step whose force evaluation is the hot path: Plummer sphere,
N = 131072 (2^17), G = 1, equal masses, seed 2, softening 1e-3, FP32
split-precision direct sum with Kahan-compensated tile sums, FP64
positions/velocities, dt = 1e-3.  Inputs are resident in HBM before the timed
region.

Printed as one JSON line:
  value      directed interactions/s = steps * N (N-1) / wall time
  roofline   dominant kernel (direct_f32): 20 flops per interaction over its
             HIP-event-timed average launch, against the MI355X FP32 vector
             peak; traffic = HBM bytes per launch from rocprofv3 --pmc; the
             measured issue rates of v_fmac_f32 / v_mul_f32 / v_rsq_f32
             (gs_issue_rates) and the ceiling they put on the kernel's
             instruction mix (6 FMA + 6 MUL/SUB + 1 rsq per 64 interactions
             per lane-wave), with the kernel's fraction of it
  accuracy   relative error vs the FP64 GPU direct sum (4096 sampled targets)
  bh         Barnes-Hut, two Plummer spheres (scale radius 1, centres 10
             apart), relative errors vs the FP64 GPU direct sum on 4096
             strided particles:
             n2e20  N = 2^20 (seed 4), theta = 0.5, monopole (the reference's
                    method): particles/s of sort + build + walk
             n2e21  N = 2^21 (seed 5): "plain" = monopole theta = 0.5,
                    and the group walk at theta = 0.5 without and with local
                    expansions; candidates meeting p99 <= 1e-3 (monopole,
                    quadrupole, group walk, group walk with quadrupoles and
                    group walk with local expansions at the largest theta
                    that does, the learned correction trained on 10^6
                    samples of seed 7);
                    "chosen" = the fastest of those; the learned correction
                    at theta = 0.8 (training times, calibration on seed 8,
                    against the quadrupole walk at 0.8, with its spot check)
  whfast     4096 planetary systems (1 star + 8 planets + U{0..2000} test
             particles), WHFast dt = 0.01, 10^4 steps: particle-steps/s of
             the batched kernel
  cpu_baseline  the reference C library (oracle/_ref) timed on this host,
             single thread (its pairwise path is serial), on a bounded
             sample; other_configs: the same library on the Leapfrog
             N=1024 run, a WHFast sample and one Barnes-Hut evaluation at
             2^20 and 2^21 (OpenMP where the reference uses it), with the
             host's CPU model, nproc and OMP_NUM_THREADS
"""
import argparse
import json
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
for p in (REPO, os.path.join(REPO, "gravity-simulator_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

import numpy as np  # noqa: E402

N_DIRECT = 1 << 17
EPS = 1e-3
DT = 1e-3
FLOPS_PER_INTERACTION = 20.0
# algorithmic HBM bytes of one FP32 direct-sum evaluation at N = 2^17: FP64
# positions and masses in (32 B per particle), FP32 source tiles out and in
# (16 B), the FP64 result out (24 B)
ALGORITHMIC_F32_BYTES = (32.0 + 16.0 + 24.0) * N_DIRECT
FP32_PEAK_TFLOPS = 157.3
FP64_PEAK_TFLOPS = 78.6
P99_TARGET = 1e-3
# HBM bytes of one direct_f32 launch at N = 2^17 per kernel shape (block,
# targets per thread, source split), from rocprofv3 --pmc FETCH_SIZE x 2.0 +
# WRITE_SIZE x 1.0 in KiB (factors from the copy kernel: 256 MiB in / out
# reads 131083 / 262144 KiB); the writes are the FP64 per-chunk partial sums
# (profiles/direct_f32_plummer_n131072.md).  A shape not measured reports
# traffic null.
DIRECT_F32_TRAFFIC_BYTES = {
    (16, 1, 4): (2.0 * 18072.4 + 12288.0) * 1024,   # 4 chunks: 12.6 MB of partial sums
    (16, 1, 0): (2.0 * 18080.9 + 24576.0) * 1024,   # automatic split, 8 chunks
}


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def host_info():
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"cpu_model": model, "nproc": os.cpu_count(), "omp_num_threads": os.environ.get("OMP_NUM_THREADS")}


def omp_threads():
    t = os.environ.get("OMP_NUM_THREADS")
    return int(t) if t and t.isdigit() else os.cpu_count()


def cpu_baseline(x, m, sample_n):
    """Reference acceleration() (pairwise, serial) on the first sample_n particles."""
    from oracle import oracle as O

    xs, ms = np.ascontiguousarray(x[:sample_n]), np.ascontiguousarray(m[:sample_n])
    if O.ref_available():
        kind = "reference"
        fn = lambda: O.ref_acceleration(xs, ms, 1, G=1.0, eps=EPS)  # noqa: E731
    else:
        kind = "port"
        fn = lambda: O.pairwise(xs, ms, G=1.0, eps=EPS)  # noqa: E731
    t0 = time.perf_counter()
    fn()
    dt = time.perf_counter() - t0
    return {"value": sample_n * (sample_n - 1) / dt, "unit": "interactions/s", "cores": 1, "kind": kind,
            "sample": f"one FP64 pairwise force evaluation of the first {sample_n} particles of the "
                      f"N=2^17 Plummer input (eps=1e-3), {dt:.1f} s"}


def cpu_baselines_other(ic, ws_systems):
    """The reference C library (oracle/_ref, compiled from its sources, OpenMP
    on) beside the other configurations, on this host: config 1 in full, a
    bounded WHFast sample, and one Barnes-Hut evaluation per size.  The
    reference's pairwise sum and Leapfrog are serial; its WHFast drift and
    accelerations and its BH walk use OpenMP (threads = OMP_NUM_THREADS)."""
    from oracle import oracle as O

    if not O.ref_available():
        return {"skipped": "oracle/_ref not built"}
    out = {}
    x, v, m = ic.plummer(1024, 1)
    t0 = time.perf_counter()
    r = O.ref_simulation(x, v, m, 1.0, 4, 1e-3, 1.0, method=1)
    dt = time.perf_counter() - t0
    out["leapfrog_n1024"] = {"value": dt / int(r[4]) * 1e3, "unit": "ms/step", "cores": 1, "kind": "reference",
                             "sample": f"FP64 pairwise + Leapfrog, Plummer N=1024 (seed 1), eps=0, dt=1e-3, "
                                       f"all {int(r[4])} steps, {dt:.1f} s"}
    log(f"cpu baseline leapfrog N=1024: {out['leapfrog_n1024']['value']:.3f} ms/step")
    off, X, V, M = ic.ensemble(4096, 3)
    P = 0
    t0 = time.perf_counter()
    for s in range(ws_systems):
        a, b = int(off[s]), int(off[s + 1])
        O.ref_simulation(X[a:b], V[a:b], M[a:b], 1.0, 10, 0.01, 100.0, method=2)
        P += b - a
    dt = time.perf_counter() - t0
    out["whfast"] = {"value": P * 10000 / dt, "unit": "particle-steps/s", "cores": omp_threads(),
                     "kind": "reference",
                     "sample": f"WHFast massless form, the first {ws_systems} systems of the 4096-system "
                               f"ensemble (seed 3, {P} particles), dt=0.01, the full 10^4 steps each, one "
                               f"launch_simulation per system, {dt:.1f} s"}
    log(f"cpu baseline whfast: {out['whfast']['value']:.3e} particle-steps/s")
    for key, n, seed in (("bh_n2e20", 1 << 20, 4), ("bh_n2e21", 1 << 21, 5)):
        x, v, m = ic.two_spheres(n, seed)
        t0 = time.perf_counter()
        O.ref_acceleration(x, m, 3, eps=EPS, theta=0.5, leaf=1)
        dt = time.perf_counter() - t0
        out[key] = {"value": n / dt, "unit": "particles/s", "cores": omp_threads(), "kind": "reference",
                    "sample": f"one Barnes-Hut evaluation (tree build serial, walk OpenMP), two Plummer "
                              f"spheres N={n} (seed {seed}), theta=0.5, leaf 1, eps=1e-3, {dt:.1f} s; the "
                              f"reference's walk as it is (leaves without monopoles, keys looked up by "
                              f"original index), so not at the accuracy of the GPU methods"}
        log(f"cpu baseline BH N={n}: {out[key]['value']:.3e} particles/s")
    return out


def timed_evals(L, sim, p, reps, kernels):
    """Average wall ms per evaluation (device-resident) and per-kernel ms."""
    sim.acceleration(p, copy=False)
    L.synchronize()
    L.timing_enable(True)
    L.timing_reset()
    t0 = time.perf_counter()
    for _ in range(reps):
        sim.acceleration(p, copy=False)
    L.synchronize()
    wall = (time.perf_counter() - t0) / reps
    parts = {}
    for k in kernels:
        ms, calls = L.timing_query(k)
        if calls:
            parts[k + "_ms"] = ms / reps
    L.timing_enable(False)
    return wall, parts


BH_KERNELS = ["tree_sort", "tree_build", "bh_walk", "learned_features", "learned_mlp", "spot_check"]


def bh_case(L, sim, n, method, theta, reps=5, label=None):
    p = L.param(method, theta=theta, eps=EPS, leaf=1)
    wall, parts = timed_evals(L, sim, p, reps, BH_KERNELS)
    nint = L.last_walk_interactions()
    med, p99, mx = sim.accel_error(p, samples=4096)
    r = {"method": label or {3: "monopole", 19: "quadrupole", 18: "learned", 20: "group",
                                 21: "group+quadrupole", 22: "group+expansions"}[method], "theta": theta,
         "particles_per_s": n / wall, "ms_per_eval": wall * 1e3, "interactions": nint,
         "median_rel": med, "p99_rel": p99, "max_rel": mx}
    r.update({k: round(v, 4) for k, v in parts.items()})
    if method == 22:
        r["expansion_ratio"] = L.get_group_expansion_ratio()
        r["expanded_pairs"] = L.last_walk_expansion_pairs()
    if "bh_walk_ms" in parts:
        r["walk_tflops"] = FLOPS_PER_INTERACTION * nint / (parts["bh_walk_ms"] / 1e3) / 1e12
    return r


def run_bh(L, ic, learned=True):
    out = {}
    # N = 2^20, the reference's method
    n4 = 1 << 20
    x, v, m = ic.two_spheres(n4, 4)
    sim = L.Sim(x, v, m, 1.0)
    out["n2e20"] = {"workload": "two Plummer spheres N=2^20 (seed 4), eps=1e-3, leaf=1",
                    "plain": bh_case(L, sim, n4, 3, 0.5), "group": bh_case(L, sim, n4, 20, 0.5)}
    sim.close()
    log(f"BH 2^20 plain: {out['n2e20']['plain']['particles_per_s']:.3e} particles/s")

    # N = 2^21: plain vs chosen at p99 <= 1e-3
    n5 = 1 << 21
    xt, vt, mt = ic.two_spheres(n5, 7)
    x, v, m = ic.two_spheres(n5, 5)
    sim = L.Sim(x, v, m, 1.0)
    res = {"workload": "two Plummer spheres N=2^21 (seed 5), eps=1e-3, leaf=1; learned correction "
                       "trained on 10^6 samples of seed 7", "p99_target": P99_TARGET}
    res["plain"] = bh_case(L, sim, n5, 3, 0.5)
    res["group"] = bh_case(L, sim, n5, 20, 0.5)
    res["group_expansion"] = bh_case(L, sim, n5, 22, 0.5)
    log(f"BH 2^21 plain theta 0.5: p99 {res['plain']['p99_rel']:.2e}; group walk "
        f"{res['group']['particles_per_s'] / res['plain']['particles_per_s']:.2f}x, p99 {res['group']['p99_rel']:.2e}; "
        f"with expansions {res['group_expansion']['particles_per_s'] / res['plain']['particles_per_s']:.2f}x, "
        f"p99 {res['group_expansion']['p99_rel']:.2e}")
    cands = []
    for th in (0.45, 0.4, 0.35, 0.3, 0.25, 0.2):
        r = bh_case(L, sim, n5, 3, th, reps=3)
        if r["p99_rel"] <= P99_TARGET:
            res["plain_at_target"] = r
            cands.append(r)
            break
    # opening angles in steps of 0.02 near where each method crosses the target
    for th in (0.6, 0.56, 0.54, 0.52, 0.5, 0.45, 0.4):
        r = bh_case(L, sim, n5, 19, th, reps=3)
        if r["p99_rel"] <= P99_TARGET:
            res["quadrupole_at_target"] = r
            cands.append(r)
            break
    for th in (0.46, 0.44, 0.42, 0.4, 0.38, 0.35, 0.3, 0.25):
        r = bh_case(L, sim, n5, 20, th, reps=3)
        if r["p99_rel"] <= P99_TARGET:
            res["group_at_target"] = r
            cands.append(r)
            break
    for th in (0.7, 0.65, 0.62, 0.6, 0.58, 0.56, 0.55, 0.5, 0.45):
        r = bh_case(L, sim, n5, 21, th, reps=3)
        if r["p99_rel"] <= P99_TARGET:
            res["group_quadrupole_at_target"] = r
            cands.append(r)
            break
    for th in (0.44, 0.42, 0.41, 0.4, 0.38, 0.35, 0.3, 0.25):
        r = bh_case(L, sim, n5, 22, th, reps=3)
        if r["p99_rel"] <= P99_TARGET:
            res["group_expansion_at_target"] = r
            cands.append(r)
            break
    log("BH 2^21 monopole / quadrupole / group / group+expansions at target done")

    if not learned:
        sim.close()
        out["n2e21"] = res
        return out
    # learned correction, the specified coarse walk (theta = 0.8): trained on
    # seed 7, output scale chosen on an independent realisation (seed 8),
    # evaluated on seed 5 against its own quadrupole sum (method 19 at 0.8)
    xv, vv, mv = ic.two_spheres(n5, 8)
    t0 = time.perf_counter()
    loss = L.learned_train(xt, mt, eps=EPS, theta=0.8, leaf=1, samples=1000000, epochs=10, batch=4096,
                           lr=3e-3, seed=5)
    train_s = time.perf_counter() - t0
    train_ms = L.learned_training_times()
    rep = L.learned_training_report()
    L.learned_calibrate(xv, mv, eps=EPS, theta=0.8, leaf=1, samples=1 << 18, seed=11)
    cal = L.learned_training_report()
    L.learned_set_policy(1.0, 0, 0.5)
    raw = bh_case(L, sim, n5, 18, 0.8, reps=3)
    quad08 = bh_case(L, sim, n5, 19, 0.8, reps=3)
    L.learned_set_policy(P99_TARGET, 1024, 0.5)
    checked = bh_case(L, sim, n5, 18, 0.8, reps=3, label="learned+spot-check")
    spot_p99, fell_back = L.learned_status()
    res["learned_theta0.8"] = {"train_s": train_s, "train_ms": train_ms, "train_loss": loss, "held_out": rep,
                               "calibration_seed8": cal, "without_check": raw,
                               "quadrupole_theta0.8": quad08,
                               "learned_over_quadrupole_p99": raw["p99_rel"] / quad08["p99_rel"],
                               "learned_over_quadrupole_median": raw["median_rel"] / quad08["median_rel"],
                               "with_check": checked, "spot_check_p99_after": spot_p99,
                               "fell_back": fell_back,
                               "fallback": "group walk with quadrupoles at theta 0.5, checked again"}
    log(f"BH 2^21 learned 0.8: p99 {raw['p99_rel']:.2e} (quadrupole 0.8: {quad08['p99_rel']:.2e}, alpha "
        f"{cal['alpha']}), fell back {fell_back}")
    # learned correction at the coarsest theta whose spot check passes
    for th in (0.55, 0.5, 0.45, 0.4):
        L.learned_train(xt, mt, eps=EPS, theta=th, leaf=1, samples=1000000, epochs=10, batch=4096, lr=3e-3,
                        seed=5)
        L.learned_calibrate(xv, mv, eps=EPS, theta=th, leaf=1, samples=1 << 18, seed=11)
        L.learned_set_policy(P99_TARGET, 1024, 0.5)
        r = bh_case(L, sim, n5, 18, th, reps=3, label="learned+spot-check")
        sp, fb = L.learned_status()
        r["spot_check_p99"], r["fell_back"] = sp, fb
        r["held_out"] = L.learned_training_report()
        if not fb and r["p99_rel"] <= P99_TARGET:
            res["learned_at_target"] = r
            cands.append(r)
            break
    L.learned_set_policy(P99_TARGET, 1024, 0.5)
    sim.close()
    if cands:
        best = max(cands, key=lambda r: r["particles_per_s"])
        res["chosen"] = {"method": best["method"], "theta": best["theta"],
                         "particles_per_s": best["particles_per_s"], "p99_rel": best["p99_rel"]}
        if "plain_at_target" in res:
            res["chosen_vs_plain_at_equal_p99"] = best["particles_per_s"] / res["plain_at_target"]["particles_per_s"]
        res["chosen_vs_plain_theta0.5"] = best["particles_per_s"] / res["plain"]["particles_per_s"]
    out["n2e21"] = res
    log(f"BH 2^21 chosen: {res.get('chosen')}")
    return out


def run_small_leapfrog(L, ic):
    """FP64 direct sum + Leapfrog at N=1024 (Plummer seed 1, eps=0, dt=1e-3,
    1000 steps), as users run it and with per-kernel events."""
    x, v, m = ic.plummer(1024, 1)
    p = L.param(1)
    out = {"workload": "FP64 pairwise + Leapfrog, Plummer N=1024 (seed 1), eps=0, dt=1e-3, 1000 steps"}
    for mode in ("plain", "with_events"):
        sim = L.Sim(x, v, m, 1.0)
        sim.leapfrog_begin(p, 1e-3)
        L.timing_enable(mode == "with_events")  # timing on -> every kernel launched with its own events
        L.synchronize()
        t0 = time.perf_counter()
        sim.leapfrog_steps(p, 1e-3, 1000)
        L.synchronize()
        wall = time.perf_counter() - t0
        L.timing_enable(False)
        sim.close()
        out[f"{mode}_ms_per_step"] = wall
    out["interactions_per_s"] = 1024 * 1023 / (out["plain_ms_per_step"] / 1000.0)
    return out


def run_integrators(L, ic):
    """Device-resident integrators through launch_simulation, Plummer N=1024
    (seed 1), eps=1e-3, FP64 pairwise forces (bitwise with the reference):
    fixed-step Euler / RK4 at dt=1e-3 to t=0.2, the adaptive DOPRI, RKF78 and
    IAS15 at tolerance 1e-9 to t=0.2; and RK4 with the FP32 split direct sum at
    N=2^17 (seed 2), 10 steps."""
    x, v, m = ic.plummer(1024, 1)
    out = {"workload": "Plummer N=1024 (seed 1), eps=1e-3, FP64 pairwise forces, to t=0.2"}
    cases = (("euler", 1, 1e-3, -1.0, 1), ("rk4", 3, 1e-3, -1.0, 4), ("dopri", 6, -1.0, 1e-9, 7),
             ("rkf78", 8, -1.0, 1e-9, 13), ("ias15", 9, -1.0, 1e-9, None))
    for name, integ, dt, tol, evals in cases:
        L.launch_simulation(x[:64], v[:64], m[:64], 1.0, integ, dt, 0.01, method=1, eps=1e-3, tolerance=tol)
        t0 = time.perf_counter()
        r = L.launch_simulation(x, v, m, 1.0, integ, dt, 0.2, method=1, eps=1e-3, tolerance=tol)
        wall = time.perf_counter() - t0
        steps = int(r[4])
        out[name] = {"steps": steps, "ms_per_step": 1e3 * wall / max(steps, 1)}
        if evals:
            out[name]["force_evals_per_s"] = steps * evals / wall
    x, v, m = ic.plummer(1 << 17, 2)
    L.launch_simulation(x[:4096], v[:4096], m[:4096], 1.0, 3, 1e-3, 2e-3, method=16, eps=1e-3)
    t0 = time.perf_counter()
    r = L.launch_simulation(x, v, m, 1.0, 3, 1e-3, 1e-2, method=16, eps=1e-3)
    wall = time.perf_counter() - t0
    out["rk4_fp32_n131072"] = {"steps": int(r[4]), "ms_per_step": 1e3 * wall / int(r[4]),
                               "interactions_per_s": 4 * int(r[4]) * float(1 << 17) * ((1 << 17) - 1) / wall}
    out["snapshots"] = run_snapshots(L, x, v, m)
    return out


def run_snapshots(L, x, v, m):
    """CSV snapshot output behind the step loop: Leapfrog with the FP32 direct
    sum at N=2^17, 64 steps of dt=2^-10, with and without a snapshot every 4
    steps (17 files of 131072 rows); and the time one synchronous snapshot of
    the same state takes on the host (what a step loop that formats in line,
    as the reference's does, pays per snapshot)."""
    import ctypes as C
    import shutil
    import tempfile
    from grav_sim_amd import _abi
    dt, tf = 2.0 ** -10, 2.0 ** -4
    t0 = time.perf_counter()
    L.launch_simulation(x, v, m, 1.0, 4, dt, tf, method=16, eps=1e-3)
    plain = time.perf_counter() - t0
    d = tempfile.mkdtemp(prefix="gs_snap_")
    try:
        t0 = time.perf_counter()
        L.launch_simulation(x, v, m, 1.0, 4, dt, tf, method=16, eps=1e-3, output_dir=d, output_interval=4 * dt)
        with_out = time.perf_counter() - t0
        files = len(os.listdir(d))
        lib = L.load()
        xs, vs, ms = (np.ascontiguousarray(a) for a in (x, v, m))
        s = _abi.make_system(xs, vs, ms, 1.0)
        op = lib.get_new_output_param()
        op.method, op.output_dir, op.output_interval = 2, (d + "/").encode(), 1.0
        op.output_count_ = 1000
        t0 = time.perf_counter()
        st = lib.output_snapshot(C.byref(op), C.byref(s), C.byref(lib.get_new_integrator_param()),
                                 C.byref(L.param(1)), C.byref(_abi.SimulationStatus()),
                                 C.byref(lib.get_new_settings()))
        sync_one = time.perf_counter() - t0
        L.check(st, "output_snapshot")
    finally:
        shutil.rmtree(d, ignore_errors=True)
    return {"workload": "Leapfrog, FP32 direct sum, Plummer N=2^17 (seed 2), 64 steps, a snapshot every 4 steps",
            "files": files, "run_s_without_output": plain, "run_s_with_output": with_out,
            "sync_snapshot_s": sync_one, "inline_formatting_s_est": files * sync_one,
            "rows_per_s_sync": len(m) / sync_one}


def pm_lattice(nside, box, seed):
    """A perturbed lattice (nside^3 particles, Gaussian displacements of 0.3
    lattice spacings) in [0, box)^3, unit total mass."""
    rng = np.random.default_rng(seed)
    q = (np.arange(nside) + 0.5) * (box / nside)
    x = np.stack(np.meshgrid(q, q, q, indexing="ij"), axis=-1).reshape(-1, 3)
    x = np.mod(x + 0.3 * (box / nside) * rng.standard_normal(x.shape), box)
    return x, np.full(len(x), 1.0 / len(x))


def run_pm(L, evals=5, cpu=True, shuffle=False):
    """Particle mesh: one force evaluation for 128^3 particles on a 256^3 grid
    (per-kernel times over `evals` evaluations), 50 steps of the
    cosmological Leapfrog (LambdaCDM, a = 0.1 -> 0.2), and the numpy
    restatement on a 64^3-particle, 64^3-grid sample as the CPU baseline.
    shuffle=True permutes the particles randomly (the arrays' order, not the
    positions)."""
    nside, grid, box = 128, 256, 100.0
    x, m = pm_lattice(nside, box, 13)
    if shuffle:
        perm = np.random.default_rng(1).permutation(len(m))
        x, m = x[perm], m[perm]
    c, bw = np.full(3, box / 2), box / 2
    rho = m.sum() / box ** 3
    H0, om, a = 70.0, 0.3, 0.5
    L.acceleration_pm(x, m, c, bw, H0, om, rho, grid, a)  # plans, buffers
    L.timing_enable(True)
    L.timing_reset()
    t0 = time.perf_counter()
    for _ in range(evals):
        L.acceleration_pm(x, m, c, bw, H0, om, rho, grid, a)
    wall = (time.perf_counter() - t0) / evals
    ks = {k: L.timing_query(k)[0] / evals for k in ("pm_deposit", "pm_fft", "pm_interp")}
    L.timing_enable(False)
    n = len(m)
    dev_ms = sum(ks.values())
    cells = float(grid) ** 3
    # algorithmic bytes: the deposit clears and fills the grid (16 B/cell) from
    # x, m (32 B/particle); the gradient + gather reads the potential once
    # (8 B/cell), x and writes a (48 B/particle)
    dep_gbs = (16.0 * cells + 32.0 * n) / (ks["pm_deposit"] * 1e-3) / 1e9
    interp_gbs = (8.0 * cells + 48.0 * n) / (ks["pm_interp"] * 1e-3) / 1e9
    L.leapfrog_cosmology(x, np.zeros_like(x), m, c, bw, 0.7, 0.3, 0.7, 0.01, 0.1, 0.11, grid)
    t0 = time.perf_counter()
    xs, steps, tt = L.leapfrog_cosmology(x, np.zeros_like(x), m, c, bw, 0.7, 0.3, 0.7, 0.002, 0.1, 0.2, grid)
    cos_ms = (time.perf_counter() - t0) / steps * 1e3
    out = {"workload": f"perturbed lattice {nside}^3 = {n} particles, {grid}^3 grid, FP64",
           "particles": n, "grid": grid, "kernel_ms": ks, "device_ms_per_eval": dev_ms,
           "particles_per_s": n / (dev_ms * 1e-3), "wall_ms_per_eval_incl_transfers": wall * 1e3,
           "deposit_gbs": dep_gbs, "grad_interp_gbs": interp_gbs,
           "cosmology_leapfrog": {"steps": int(steps), "ms_per_step": cos_ms}}
    if cpu:
        sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
        from oracle import pm as P
        xs, ms = pm_lattice(64, box, 14)
        t0 = time.perf_counter()
        P.acceleration_pm(xs, ms, c, bw, H0, om, ms.sum() / box ** 3, 64, a)
        cpu_s = time.perf_counter() - t0
        L.acceleration_pm(xs, ms, c, bw, H0, om, ms.sum() / box ** 3, 64, a)
        t0 = time.perf_counter()
        L.acceleration_pm(xs, ms, c, bw, H0, om, ms.sum() / box ** 3, 64, a)
        gpu_s = time.perf_counter() - t0
        out["cpu_baseline"] = {"kind": "port", "cores": 1, "sample": "64^3 particles, 64^3 grid (numpy restatement)",
                               "cpu_s": cpu_s, "gpu_wall_s_same_sample": gpu_s,
                               "cpu_particles_per_s": len(ms) / cpu_s}
    return out


def run_whfast(L, ic, steps):
    off, X, V, M = ic.ensemble(4096, 3)
    P = int(off[-1])
    counts = np.diff(off)
    T = counts - 9
    dt = 0.01
    L.timing_enable(True)
    L.timing_reset()
    t0 = time.perf_counter()
    L.whfast_ensemble(off, X, V, M, 1.0, dt, steps * dt, method=2)
    wall = time.perf_counter() - t0
    k_ms, k_calls = L.timing_query("whfast_steps")
    i_ms, _ = L.timing_query("whfast_init")
    L.timing_enable(False)
    # 20 flops per pair force (massive-massive and massive-test) + 150 flops
    # per Kepler drift, per system-step
    flops = steps * float(np.sum(20.0 * (9 * 8 + 9 * T) + 150.0 * (counts - 1)))
    return {"workload": f"4096 systems (1 star + 8 planets + U{{0..2000}} test particles, seed 3), "
                        f"{P} particles, WHFast dt=0.01, {steps} steps, massless form",
            "particles": P, "steps": steps,
            "particle_steps_per_s": P * steps / (k_ms / 1e3), "kernel_ms": k_ms, "init_ms": i_ms,
            "wall_s_incl_transfers": wall,
            "fp64_tflops": flops / (k_ms / 1e3) / 1e12, "fp64_frac": flops / (k_ms / 1e3) / 1e12 / FP64_PEAK_TFLOPS}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--cpu-sample", type=int, default=90000)
    ap.add_argument("--whfast-steps", type=int, default=10000)
    ap.add_argument("--cpu-whfast-systems", type=int, default=16)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-bh", action="store_true")
    ap.add_argument("--no-whfast", action="store_true")
    ap.add_argument("--no-pm", action="store_true", help="skip the particle-mesh leg")
    ap.add_argument("--pm-shuffle", action="store_true",
                    help="particle-mesh leg with the lattice's particles in random order")
    ap.add_argument("--no-learned", action="store_true", help="Barnes-Hut without the learned correction")
    ap.add_argument("--no-integrators", action="store_true")
    ap.add_argument("--no-autotune", action="store_true",
                    help="skip the FP32 shape autotuner (default: it runs first and picks the shape)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU (asked for --gpus {args.gpus}): this build runs on a single "
              "MI355X; the multi-GPU decomposition is described, not built", file=sys.stderr)
        sys.exit(2)

    from grav_sim_amd import ic
    from grav_sim_amd import lib as L

    info = L.device_info()
    x, v, m = ic.plummer(N_DIRECT, 2)
    # the HBM copy calibration first: the autotuner's FP32 load then runs
    # right before the timed region, so the clocks are up when it starts
    copy_gbs = L.copy_calibrate(1 << 28, 5)
    # FP32 issue rates (cycles per wave64 instruction, measured at the
    # device's nominal clock) of the instruction forms the kernels use
    issue = L.issue_rates()
    simd_cycles_per_s = 4.0 * info.cu_count * info.clock_khz * 1e3
    fma_peak = simd_cycles_per_s * 64 * 2 / issue["fma"] / 1e12
    # the direct-sum interaction (counters: 13.1 VALU wave-instructions per 64
    # interactions): 6 FMA, 6 MUL/SUB and one v_rsq_f32 per lane
    mix_cycles = 6 * issue["fma"] + 6 * issue["mul"] + issue["rsq"]
    mix_ceiling = simd_cycles_per_s * 64 * FLOPS_PER_INTERACTION / mix_cycles / 1e12
    log(f"issue: fma {issue['fma']:.2f}, mul {issue['mul']:.2f}, rsq {issue['rsq']:.2f} cycles per wave64 "
        f"instruction; FMA chains {fma_peak:.1f} TFLOP/s; direct-sum mix ceiling {mix_ceiling:.1f} TFLOP/s")
    tune = None
    if not args.no_autotune:
        t0 = time.perf_counter()
        b, i, sp = L.autotune_fp32(N_DIRECT)
        tune = {"block": b, "targets_per_thread": i, "source_split": sp, "autotune_s": time.perf_counter() - t0}
        log(f"autotuner: block {b}, targets/thread {i}, split {sp} ({tune['autotune_s']:.1f} s)")
    else:
        b, i, sp = L.get_fp32_config()
        tune = {"block": b, "targets_per_thread": i, "source_split": sp, "autotune_s": None}
    p = L.param(16, eps=EPS)
    sim = L.Sim(x, v, m, 1.0)
    sim.leapfrog_begin(p, DT)
    sim.leapfrog_steps(p, DT, args.warmup)
    L.synchronize()
    L.timing_enable(True)
    L.timing_reset()
    t0 = time.perf_counter()
    sim.leapfrog_steps(p, DT, args.steps)
    L.synchronize()
    wall = time.perf_counter() - t0
    ms, calls = L.timing_query("direct_f32")
    L.timing_enable(False)
    inter = float(N_DIRECT) * (N_DIRECT - 1)
    value = args.steps * inter / wall
    kavg = ms / max(calls, 1) / 1e3
    achieved = FLOPS_PER_INTERACTION * inter / kavg / 1e12
    med, p99, mx = sim.accel_error(p, samples=4096)
    sim.close()
    log(f"direct: {value:.4e} interactions/s, kernel {kavg * 1e3:.3f} ms, {achieved:.1f} TFLOP/s")

    out = {
        "metric": "interactions/s + BH particles/s at fixed accel error vs FP64; plain vs chosen",
        "value": value,
        "unit": "interactions/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": wall / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {"workload": "FP32 split-precision direct sum + Leapfrog, Plummer N=131072, seed 2, "
                               "eps=1e-3, dt=1e-3", "N": N_DIRECT, "fp32_shape": tune},
        "roofline": {"bound": "fp32-valu", "achieved": achieved, "peak": FP32_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": achieved / FP32_PEAK_TFLOPS,
                     "traffic": DIRECT_F32_TRAFFIC_BYTES.get((tune["block"], tune["targets_per_thread"],
                                                              tune["source_split"])),
                     "algorithmic_bytes": ALGORITHMIC_F32_BYTES,
                     "kernel": "direct_f32", "kernel_avg_ms": kavg * 1e3,
                     "flops_per_launch": FLOPS_PER_INTERACTION * inter,
                     "fp32_issue_cycles": issue,
                     "measured_fma_peak": fma_peak,
                     "frac_of_measured_fma_peak": achieved / fma_peak,
                     "instruction_mix_ceiling": mix_ceiling,
                     "frac_of_instruction_mix_ceiling": achieved / mix_ceiling},
        "accuracy": {"vs": "FP64 GPU direct sum, 4096 sampled targets", "median_rel": med, "p99_rel": p99,
                     "max_rel": mx},
        "hbm_copy_gbs": copy_gbs,
        "device": {"name": info.name.decode(), "arch": info.arch.decode(), "cu": info.cu_count,
                   "clock_khz": info.clock_khz},
    }
    if not args.no_bh:
        out["bh"] = run_bh(L, ic, learned=not args.no_learned)
    out["leapfrog_n1024"] = run_small_leapfrog(L, ic)
    if not args.no_integrators:
        out["integrators"] = run_integrators(L, ic)
        log("integrators: " + ", ".join(f"{k} {v['ms_per_step']:.3f} ms/step" for k, v in out["integrators"].items()
                                        if isinstance(v, dict) and "ms_per_step" in v))
        sn = out["integrators"]["snapshots"]
        log(f"snapshots: {sn['files']} files, run {sn['run_s_with_output']:.3f} s with output vs "
            f"{sn['run_s_without_output']:.3f} s without; one synchronous snapshot {sn['sync_snapshot_s']:.3f} s")
    log(f"leapfrog N=1024: {out['leapfrog_n1024']['plain_ms_per_step']:.4f} ms/step, "
        f"with events {out['leapfrog_n1024']['with_events_ms_per_step']:.4f} ms/step")
    if not args.no_whfast:
        out["whfast"] = run_whfast(L, ic, args.whfast_steps)
        log(f"whfast: {out['whfast']['particle_steps_per_s']:.3e} particle-steps/s")
    if not args.no_pm:
        out["pm"] = run_pm(L, cpu=not args.no_cpu, shuffle=args.pm_shuffle)
        log(f"pm: {out['pm']['particles_per_s']:.3e} particles/s ({out['pm']['device_ms_per_eval']:.3f} ms per "
            f"evaluation), cosmological Leapfrog {out['pm']['cosmology_leapfrog']['ms_per_step']:.3f} ms/step")
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(x, m, args.cpu_sample)
        out["cpu_baseline"]["host"] = host_info()
        out["cpu_baseline"]["other_configs"] = cpu_baselines_other(ic, args.cpu_whfast_systems)
        oc = out["cpu_baseline"]["other_configs"]
        ratios = {}
        if "leapfrog_n1024" in oc:
            ratios["leapfrog_n1024"] = oc["leapfrog_n1024"]["value"] / out["leapfrog_n1024"]["plain_ms_per_step"]
        if "whfast" in oc and "whfast" in out:
            ratios["whfast"] = out["whfast"]["particle_steps_per_s"] / oc["whfast"]["value"]
        if "bh_n2e20" in oc and "bh" in out:
            ratios["bh_n2e20_plain"] = out["bh"]["n2e20"]["plain"]["particles_per_s"] / oc["bh_n2e20"]["value"]
        if "bh_n2e21" in oc and "bh" in out and "chosen" in out["bh"]["n2e21"]:
            ratios["bh_n2e21_chosen"] = out["bh"]["n2e21"]["chosen"]["particles_per_s"] / oc["bh_n2e21"]["value"]
        oc["gpu_over_cpu"] = ratios
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
