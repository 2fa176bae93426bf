#!/usr/bin/env python3
"""Benchmark of the DEM time step on one MI355X.

Workload: the superquadric bed -- 1,000,000 superquadrics (semi-axes
U[0.4, 1] mm, blockiness n1, n2 U[2, 8], random orientations, solid fraction
0.3, periodic in x and y with floor and ceiling walls, Hooke kn = 1e5,
en = 0.8, mu = 0.3, dt = 1e-6, at rest under gravity).  A "step" is one
iteration of the reference driver loop (Grains/Base/src/GrainsCPU.cpp:55-66):
broad phase, narrow phase + contact force, gravity, integration.

Prints ONE JSON line: particle-steps/s of the FP32-mixed path (value), the
plain FP64 path beside it, the FP32-mixed position error against FP64 after
the same steps, GJK pair tests/s (in the step and on the reference's GJK
microbenchmark), the roofline of the dominant kernel measured with HIP events
over the timed region, and the FP64 CPU oracle timed on this host.

--workload selects another workload, with a line of the same form:
c0 the reference's 1,000-sphere walled box (FP64, 1,000 steps), c2 polydisperse polyhedra (250k cubes, hulls and spheres, 2,000 steps at
dt = 5e-7), c3 the batched ensemble (512 beds, ~2.7M particles, autotuned
launch, one graph), c4 the differentiable calibration (8,192 spheres and
ellipsoids, forward + adjoint gradients against finite differences).
"""
import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

from grains3dgpu_amd import _abi as A  # noqa: E402
from grains3dgpu_amd import scene as S  # noqa: E402

PEAK_HBM_GBS = 8000.0
PEAK_FP32_TFLOPS = 157.3
PEAK_FP64_TFLOPS = 78.6
# Algorithmic operations of the narrow-phase kernel, counted from the source
# (gr_geom.hpp; transcendental = 1 op, FMA = 2 ops): one GJK iteration = two
# log-domain superquadric supports (2 x 42), the rotation of the direction
# into B's frame and of B's support into A's, with the unit-frame scaling
# (42), lower bound, separation and gap tests (10), the signed-volume
# sub-algorithm (segment 20, triangle 64 + its edge fall-backs, tetrahedron
# 62 + its face fall-backs: ~80 on average over the simplex sizes met) and
# |v| (6).
OPS_PER_GJK_ITER = 222
# per pair reaching GJK: two rotation matrices (2 x 30), the relative
# transform (63), OBB test (110), support set-up (2 x 16), witness points and
# contact vector (45), Hooke force when in contact (counted always, 80)
OPS_PER_GJK_PAIR = 390
# per candidate entry: loads, periodic image, bounding-sphere test (20)
OPS_PER_ENTRY = 20
# Compulsory HBM bytes of one narrow-phase launch (k_screen): each particle's
# pose (pos 24 + quat 32, FP64) and shape and sim ids (8) once, each shape's
# narrow-phase record (ShapeNP<float>, 96) once, each candidate entry's two
# ids (8) and flag (4), each contact's force and torque (FP32, 24)
B_NP_PARTICLE = 64
B_NP_SHAPE = 96
B_NP_ENTRY = 12
B_NP_CONTACT = 24
# warm-started GJK: the pair's previous direction record (16 B) read and the
# new one written, per candidate entry, plus each particle's record count
B_NP_WARM_ENTRY = 32
B_NP_WARM_PARTICLE = 8
# Compulsory HBM bytes of one step's integration: each particle's pose (64) and
# velocity (48) records read and written, the position its lists were built
# at (32), its shape's dynamics (64), its entries' offset and marks (12);
# each candidate entry's flag (4); each contact's force and torque (24)
B_INT_PARTICLE = 332
B_INT_ENTRY = 4
B_INT_CONTACT = 24
# Compulsory HBM bytes per particle-step: the pose and velocity records read
# and written (112 + 112); FP64 reads an FP64 shape record more of
B_PS_FP32 = 224
B_PS_FP64 = 272


def log(*a):
    print(*a, file=sys.stderr, flush=True)


# GJK relative tolerances of the superquadric bed workload: 1e-10 (FP64),
# 1e-6 (FP32)
GJK_TOL = {A.FP64: 1e-10, A.FP32_MIXED: 1e-6}

# FP32-mixed runs start each pair's GJK search from the pair's direction of
# the previous step (GRAINS_WARM_START; the cold start is timed beside it)
# and take the geometry of the pairs in contact from an FP64 re-run
# (GRAINS_FP64_CONTACTS; FP32 contact geometry is measured beside it)
FP32_FLAGS = A.WARM_START | A.FP64_CONTACTS
FP32_FLAGS_FP32_CONTACTS = A.WARM_START


MAX_STATS = ("max_candidates", "gjk_max_iterations", "sort_passes", "fp64_refine_max_iterations")

# --eager: timed steps launched kernel by kernel, not replayed from a graph
EAGER = False


def run_engine(sc, precision, warmup, steps, profile=True, flags=0, gjk_tol=None, graph=True, profile_steps=100,
               max_neighbors=64, graph_steps=1, **launch):
    """W warm-up steps as the timed ones are launched (their graphs are captured
    here), then (profile) min(profile_steps, steps) eagerly
    launched steps with HIP events around every phase, then `steps` timed
    steps replayed from a captured graph (the production mode).  Returns the
    timed wall time, the counters of the timed steps and per-step phase
    times.  `launch`: block_size, narrow_blocks_per_cu, narrow_passes;
    graph_steps: steps captured in one graph."""
    from grains3dgpu_amd.engine import Engine
    tol = GJK_TOL[precision] if gjk_tol is None else gjk_tol
    e = S.load(Engine(dt=sc.dt, precision=precision, max_neighbors=max_neighbors, gjk_rel_tol=tol, flags=flags,
                      **launch), sc)
    e.set_graph_steps(graph_steps)
    graph = graph and not EAGER
    if warmup:
        e.step(warmup, graph=graph)
    phases = None
    if profile:
        kp = min(profile_steps, steps)
        e.set_profiling(True)
        e.step(kp)
        phases = {p: v / kp for p, v in e.get_phase_times().items()}
        e.set_profiling(False)
        log(f"    {kp} profiled steps: {', '.join(f'{p} {v:.3f}' for p, v in phases.items())} ms")
    # timed in at most 10 chunks so a long run keeps reporting progress
    chunk = max(100, -(-steps // 10))
    done, wall, stats = 0, 0.0, None
    while done < steps:
        k = min(chunk, steps - done)
        t0 = time.perf_counter()
        e.step(k, graph=graph)
        wall += time.perf_counter() - t0
        st = e.get_stats()
        stats = st if stats is None else {c: (max(stats[c], st[c]) if c in MAX_STATS else stats[c] + st[c])
                                          for c in st}
        done += k
        log(f"    {done}/{steps} steps, {wall:.2f} s")
    pos, quat, vel, om = e.get_state()
    e.close()
    return dict(wall_s=wall, stats=stats, phases=phases, pos=pos, vel=vel)


def testdev_pairs(n_pairs=614_400, seed=0):
    """The reference's GJK microbenchmark workload (GrainsTestDev.cpp:75-141):
    superquadrics r = 0.05, n1 = n2 = 3; centres N(-0.05, 0.005) and
    N(+0.05, 0.005) per axis; random Euler angles U[0, 2 pi)."""
    rng = np.random.default_rng(seed)

    def basis(ang):
        ax, ay, az = ang.T
        cx, sx, cy, sy, cz, sz = np.cos(ax), np.sin(ax), np.cos(ay), np.sin(ay), np.cos(az), np.sin(az)
        m = np.stack([cz * cy, cz * sy * sx - sz * cx, cz * sy * cx + sz * sx,
                      sz * cy, sz * sy * sx + cz * cx, sz * sy * cx - cz * sx,
                      -sy, cy * sx, cy * cx], 1)
        return m   # Transform3::setBasis(aX, aY, aZ) (Transform3.cpp:151-162)

    ta = np.concatenate([basis(rng.uniform(0, 2 * math.pi, (n_pairs, 3))),
                         rng.normal(-0.05, 0.005, (n_pairs, 3))], 1)
    tb = np.concatenate([basis(rng.uniform(0, 2 * math.pi, (n_pairs, 3))),
                         rng.normal(0.05, 0.005, (n_pairs, 3))], 1)
    return ta, tb


def gjk_microbench(precision):
    from grains3dgpu_amd.engine import Engine
    ta, tb = testdev_pairs()
    n = len(ta)
    e = Engine(precision=precision, flags=A.REF_QUIRKS)
    shp = S.Scene(shapes=[dict(kind=A.SUPERQUADRIC, dims=(0.05, 0.05, 0.05, 3.0, 3.0), density=1.0)],
                  tables=np.array([S.hooke_row(1e5, 0.8, 0, 0.3)]), n_materials=1,
                  sims=[dict(domain_min=(0, 0, 0), domain_max=(1, 1, 1))],
                  particle_shape=np.zeros(1, np.uint32), pos=np.zeros((1, 3)),
                  quat=np.array([[0, 0, 0, 1.0]]), vel=np.zeros((1, 3)), omega=np.zeros((1, 3)))
    e.set_shapes(shp)
    z = np.zeros(n, np.uint32)
    e.gjk_batch(z, z, ta, tb)          # warm-up
    d, _, _, it = e.gjk_batch(z, z, ta, tb)
    ms = e.gjk_batch_kernel_ms()
    e.close()
    return dict(pairs=n, kernel_ms=ms, pair_tests_per_s=n / (ms * 1e-3), mean_iterations=float(it.mean()),
                finite=bool(np.isfinite(d).all()))


def copy_calibration(nbytes=1 << 30, reps=3):
    """A plain copy kernel of known size: each dispatch reads and writes
    nbytes.  FETCH_SIZE / WRITE_SIZE per dispatch of this run, divided by
    nbytes / 1024, give the factors that turn the counters of the step's
    kernels into HBM bytes."""
    import torch
    a = torch.ones(nbytes // 4, dtype=torch.float32, device="cuda")
    b = torch.empty_like(a)
    for _ in range(reps):
        b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes_per_dispatch": nbytes, "dispatches": reps}), flush=True)


def shape_bytes(sc):
    """Narrow-phase shape records (ShapeNP<float>, 96 B) of the shapes the
    particles use, plus their polyhedron vertices (FP32, 12 B each)."""
    used = np.unique(sc.particle_shape)
    nv = 0
    if len(sc.vertices):
        sh = sc.shapes
        nv = int(sum(int(sh[int(k)]["n_vertices"]) for k in used))
    return len(used) * B_NP_SHAPE + 12 * nv


def measured_traffic(traffic_file):
    """HBM bytes per launch by kernel, from the FETCH_SIZE and WRITE_SIZE
    counter runs summarised in profiles/ (lines "hbm_bytes_per_launch
    <kernel> = N"); empty until measured."""
    out = {}
    tf = os.path.join(ROOT, "profiles", traffic_file) if traffic_file else None
    if tf and os.path.exists(tf):
        for line in open(tf):
            if line.strip().startswith("hbm_bytes_per_launch"):
                key, val = line.split("=")
                out[key.split()[1]] = float(val)
    return out


def narrow_roofline(sc, r, K, traffic=None, warm=True):
    """Roofline of the screening narrow pass (k_screen<float,warm>,
    one launch per step): compulsory bytes per launch over its HIP-event
    time."""
    st = r["stats"]
    nar_ms = r["phases"]["narrow"]
    E, C = st["candidate_pairs"] / K, st["contacts"] / K
    nbytes = sc.n * B_NP_PARTICLE + shape_bytes(sc) + E * B_NP_ENTRY + C * B_NP_CONTACT
    if warm:
        nbytes += E * B_NP_WARM_ENTRY + sc.n * B_NP_WARM_PARTICLE
    achieved_gbs = nbytes / (nar_ms * 1e-3) / 1e9
    kernel = "k_screen<float,true>" if warm else "k_screen<float,false>"
    return dict(bound="hbm", kernel=kernel, achieved=achieved_gbs, peak=PEAK_HBM_GBS,
                unit="GB/s", frac=achieved_gbs / PEAK_HBM_GBS, traffic=(traffic or {}).get(kernel),
                bytes_per_launch=nbytes, avg_launch_ms=nar_ms,
                note="screening narrow pass (every candidate entry); compulsory bytes: 64 B pose+ids per "
                     "particle, 96 B per shape record (+12 B per polyhedron vertex), 12 B per candidate "
                     "entry, 24 B per contact" + (", 32 B per entry and 8 B per particle of warm-start "
                                                   "records" if warm else "") + "; the launch is gather-latency bound")


def integrate_roofline(sc, r, K, traffic=None):
    """Roofline of the integration (k_integrate and the queues of particles
    near obstacles): compulsory bytes per step over its HIP-event time."""
    st = r["stats"]
    ms = r["phases"]["integrate"]
    nbytes = sc.n * B_INT_PARTICLE + st["candidate_pairs"] / K * B_INT_ENTRY + st["contacts"] / K * B_INT_CONTACT
    achieved_gbs = nbytes / (ms * 1e-3) / 1e9
    kernel = "k_integrate<float,false>"
    return dict(bound="hbm", kernel=kernel, achieved=achieved_gbs, peak=PEAK_HBM_GBS, unit="GB/s",
                frac=achieved_gbs / PEAK_HBM_GBS, traffic=(traffic or {}).get(kernel),
                bytes_per_launch=nbytes, avg_launch_ms=ms,
                note="integration; compulsory bytes: 332 B per particle (records read and written, dynamics, list "
                     "position), 4 B per candidate entry, 24 B per contact")


def valu_roofline(r, K):
    st = r["stats"]
    ops = OPS_PER_GJK_ITER * st["gjk_iterations"] / K + OPS_PER_GJK_PAIR * st["gjk_calls"] / K + \
        OPS_PER_ENTRY * st["candidate_pairs"] / K
    nar_all_ms = r["phases"]["narrow"] + r["phases"]["narrow_deferred"]
    achieved = ops / (nar_all_ms * 1e-3) / 1e12
    return dict(bound="valu", kernel="k_screen<float>, k_complete<float>", achieved=achieved, peak=PEAK_FP32_TFLOPS,
                unit="TFLOP/s", frac=achieved / PEAK_FP32_TFLOPS, ops_per_launch=ops,
                note="no MFMA: no dense contraction on the path; peak = FP32 vector")


def pos_error(run, ref, pos0, sc=None):
    """Errors of `run` against `ref` (dicts with pos, vel), with minimum-image
    differences along the periodic sides of sc's first sim:
    pos_rel_displacement = max_i |x_i - x_i^ref| / max_i |x_i^ref - x_i^0|,
    vel_rel = max_i |v_i - v_i^ref| / max_i |v_i^ref|,
    pos_rel = max_i |x_i - x_i^ref| / |x_i^ref| (the per-particle relative
    position error), pos_rel_box = max_i |x_i - x_i^ref| / the box diagonal."""
    L = per = None
    if sc is not None:
        L = np.array(sc.sims[0]["domain_max"]) - np.array(sc.sims[0]["domain_min"])
        per = [(sc.sims[0].get("periodic", 0) >> k) & 1 for k in range(3)]

    def wrap(d):
        if L is not None:
            for k in range(3):
                if per[k]:
                    d[:, k] -= L[k] * np.rint(d[:, k] / L[k])
        return d

    dx = np.linalg.norm(wrap(run["pos"] - ref["pos"]), axis=1)
    disp = np.linalg.norm(wrap(ref["pos"] - pos0), axis=1).max()
    dv = np.linalg.norm(run["vel"] - ref["vel"], axis=1)
    out = dict(pos_rel_displacement=float(dx.max() / max(disp, 1e-300)),
               vel_rel=float(dv.max() / max(np.linalg.norm(ref["vel"], axis=1).max(), 1e-300)),
               pos_rel=float((dx / np.linalg.norm(ref["pos"], axis=1)).max()),
               max_displacement_m=float(disp), max_position_error_m=float(dx.max()))
    if L is not None:
        out["pos_rel_box"] = float(dx.max() / np.linalg.norm(L))
    return out


def accuracy_1000(sc, steps=1000, log=log):
    """The FP32-mixed path's error after a fixed number of steps (1,000)
    against the FP64 path (GJK 1e-10; its contact decisions and forces equal
    the FP64 oracle's, pinned by the parity tests), on a contact-bearing
    bed, with two floors beside it: the FP64 path stopped at the FP32 path's
    GJK gap 1e-6, and the FP64 path from initial positions moved by one ulp
    (the flow's own sensitivity)."""
    a32 = run_engine(sc, A.FP32_MIXED, 0, steps, profile=False, flags=FP32_FLAGS)
    f32 = run_engine(sc, A.FP32_MIXED, 0, steps, profile=False, flags=FP32_FLAGS_FP32_CONTACTS)
    a64 = run_engine(sc, A.FP64, 0, steps, profile=False)
    g64 = run_engine(sc, A.FP64, 0, steps, profile=False, gjk_tol=GJK_TOL[A.FP32_MIXED])
    sp = S.Scene(**{**sc.__dict__, "pos": np.nextafter(sc.pos, np.inf)})
    u64 = run_engine(sp, A.FP64, 0, steps, profile=False)
    err = dict(steps=steps, n=sc.n, contacts_fp64=a64["stats"]["contacts"], contacts_fp32=a32["stats"]["contacts"],
               fp64_refines_per_step=a32["stats"]["fp64_refines"] / steps,
               fp64_near_refines_per_step=a32["stats"]["fp64_near_refines"] / steps,
               **pos_error(a32, a64, sc.pos, sc),
               fp32_contact_geometry=dict(contacts=f32["stats"]["contacts"], **pos_error(f32, a64, sc.pos, sc)),
               floor_fp64_at_fp32_gap=pos_error(g64, a64, sc.pos, sc),
               floor_fp64_one_ulp=pos_error(u64, a64, sc.pos, sc))
    log(f"  FP32-mixed vs FP64 after {steps} steps: disp {err['pos_rel_displacement']:.3e}, "
        f"vel {err['vel_rel']:.3e}, per-particle {err['pos_rel']:.3e} (FP32 contact geometry: disp "
        f"{err['fp32_contact_geometry']['pos_rel_displacement']:.3e}, per-particle "
        f"{err['fp32_contact_geometry']['pos_rel']:.3e}); floors: gap "
        f"{err['floor_fp64_at_fp32_gap']['pos_rel_displacement']:.3e}, one ulp "
        f"{err['floor_fp64_one_ulp']['pos_rel_displacement']:.3e}")
    return err


def step_stats(st):
    return {k: st[k] for k in ("candidate_pairs", "gjk_calls", "gjk_iterations", "contacts", "wall_contacts",
                               "fp64_refines", "fp64_near_refines", "max_candidates", "sort_passes",
                               "out_of_domain", "nonfinite_states", "narrow_deferred", "gjk_max_iterations",
                               "fp64_refine_iterations", "fp64_refine_max_iterations")}


def host_cores():
    """Cores this process may use, capped at 16 (one GPU's share of a box)."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(16, n))


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def oracle_rate(sc, seconds, threads=1):
    """FP64 CPU oracle on scene sc for about `seconds`: particle-steps/s."""
    from oracle import pyoracle
    o = S.load(pyoracle.Oracle(dt=sc.dt, threads=threads, gjk_rel_tol=GJK_TOL[A.FP64]), sc)
    t0 = time.perf_counter()
    o.step(1)
    one = time.perf_counter() - t0
    k = max(1, int(seconds / max(one, 1e-6)))
    t0 = time.perf_counter()
    o.step(k)
    dt = time.perf_counter() - t0
    st = o.get_stats()
    o.close()
    return dict(value=sc.n * k / dt, steps=k, seconds=dt, n=sc.n, gjk_pair_tests_per_s=st["gjk_calls"] / 2 / dt)


def cpu_baseline(sc, seconds, what):
    """The FP64 oracle (same algorithm and loop order as the reference CPU
    path, OpenMP over particles) on a bounded sample: one thread (the
    reference is single-threaded) and every core of this process's share."""
    n_cores = host_cores()
    log(f"CPU baseline: FP64 oracle on {what}, {n_cores} threads and 1 thread, ~{seconds:.0f} s each")
    cm = oracle_rate(sc, seconds, threads=n_cores)
    c1 = oracle_rate(sc, seconds, threads=1)
    log(f"  {cm['value']:.3e} particle-steps/s ({n_cores} threads), {c1['value']:.3e} (1 thread)")
    return dict(value=cm["value"], unit="particle-steps/s", cores=n_cores, kind="port", cpu_model=cpu_model(),
                sample=f"{what}, {cm['n']} particles, {cm['steps']} steps in {cm['seconds']:.1f} s",
                gjk_pair_tests_per_s=cm["gjk_pair_tests_per_s"],
                single_thread=dict(value=c1["value"], steps=c1["steps"], seconds=c1["seconds"],
                                   gjk_pair_tests_per_s=c1["gjk_pair_tests_per_s"]))


def contract(metric, value, K, W, ms, dtype, workload, **extra):
    out = {"metric": metric, "value": value, "unit": "particle-steps/s", "n_gpus": 1, "steps": K, "warmup": W,
           "ms_per_step": ms, "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": dtype,
           "data": "synthetic", "config": workload}
    out.update(extra)
    return out


def bench_c1(args):
    K = args.steps or 1000
    W = args.warmup
    n = args.n or 1_000_000
    log(f"generating the superquadric bed, n = {n}")
    t0 = time.perf_counter()
    sc = S.config1(n=n, log=log)
    log(f"  done in {time.perf_counter() - t0:.1f} s: phi = {sc.notes['phi']:.4f}, "
        f"random sequential addition in {sc.notes['rounds']} rounds")

    log(f"FP32-mixed: {W} warm-up + profiled + {K} timed steps")
    # a few residents per cell: the direct candidate search (what the
    # automatic choice takes here)
    r32 = run_engine(sc, A.FP32_MIXED, W, K, flags=FP32_FLAGS, candidate_staging=1)
    ps32 = sc.n * K / r32["wall_s"]
    log(f"  {r32['wall_s'] * 1e3 / K:.3f} ms/step, {ps32:.3e} particle-steps/s")
    log(f"FP32-mixed, cold GJK starts: {W} warm-up + {K} timed steps")
    r32c = run_engine(sc, A.FP32_MIXED, W, K, profile=False, flags=A.FP64_CONTACTS, candidate_staging=1)
    log(f"  {r32c['wall_s'] * 1e3 / K:.3f} ms/step")
    r64 = None
    K64 = args.fp64_steps or K
    if not args.no_fp64:
        log(f"FP64: {W} warm-up + profiled + {K64} timed steps")
        r64 = run_engine(sc, A.FP64, W, K64)
        log(f"  {r64['wall_s'] * 1e3 / K64:.3f} ms/step")

    # errors after a fixed 1,000 steps, whatever --steps is: the bed itself
    # (at rest under gravity: grains fall ~5 um, few touch), and the same
    # distributions agitated (100k grains, velocities N(0, 0.1 m/s), angular
    # velocities N(0, 100 rad/s): collisions throughout) with its floors
    err = agit = None
    if not args.no_fp64:
        log("errors after 1,000 steps: the bed, FP32-mixed and FP64")
        e32 = run_engine(sc, A.FP32_MIXED, 0, 1000, profile=False, flags=FP32_FLAGS)
        e64 = run_engine(sc, A.FP64, 0, 1000, profile=False)
        err = dict(steps=1000, contacts_fp64=e64["stats"]["contacts"], contacts_fp32=e32["stats"]["contacts"],
                   **pos_error(e32, e64, sc.pos, sc))
        na = min(n, 100_000)
        sa = S.config1(n=na, seed=11)
        rng = np.random.default_rng(12)
        sa.vel = rng.normal(0.0, 0.1, (na, 3))
        sa.omega = rng.normal(0.0, 100.0, (na, 3))
        log(f"errors after 1,000 steps: the agitated bed, {na} particles")
        agit = accuracy_1000(sa)

    # the dominant kernel's roofline: the screening narrow pass or the
    # integration, whichever takes longer per step (the list builds, the
    # candidate search among them, serve several steps each)
    traffic = measured_traffic("step_c1_1M_traffic.txt")
    roof_int = integrate_roofline(sc, r32, K, traffic)
    roof_nar = narrow_roofline(sc, r32, K, traffic)
    roofline, roof_other = ((roof_nar, roof_int) if r32["phases"]["narrow"] >= r32["phases"]["integrate"]
                            else (roof_int, roof_nar))
    step_ms = r32["wall_s"] * 1e3 / K
    roofline_step = dict(bound="hbm", bytes_per_particle_step=B_PS_FP32,
                         achieved=B_PS_FP32 * ps32 / 1e9, peak=PEAK_HBM_GBS, unit="GB/s",
                         frac=B_PS_FP32 * ps32 / 1e9 / PEAK_HBM_GBS)

    log("GJK microbenchmark (614,400 superquadric pairs, GrainsTestDev workload)")
    mb64 = gjk_microbench(A.FP64)
    mb32 = gjk_microbench(A.FP32_MIXED)
    log(f"  FP64 {mb64['pair_tests_per_s']:.3e} /s, FP32 {mb32['pair_tests_per_s']:.3e} /s")

    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(S.config1(n=8000, seed=7), args.cpu_seconds,
                           "a superquadric bed of the same distributions and solid fraction")

    st = r32["stats"]
    out = contract(
        "particle-steps/s (FP32-mixed) on the superquadric bed", ps32, K, W, step_ms, "f32",
        {"workload": f"c1 superquadric bed: {sc.n} superquadrics a,b,c~U[0.4,1] mm, n1,n2~U[2,8], "
                     f"phi={sc.notes['phi']:.3f} by random sequential addition, periodic x,y + floor/ceiling, "
                     "dt=1e-6, at rest",
         "n_particles": sc.n, "phi": sc.notes["phi"],
         "precision": "FP32-mixed (FP64 state; FP64 geometry of the pairs in contact)"},
        fp64=None if r64 is None else {
            "particle_steps_per_s": sc.n * K64 / r64["wall_s"], "ms_per_step": r64["wall_s"] * 1e3 / K64,
            "gjk_pair_tests_per_s": r64["stats"]["gjk_calls"] / 2 / r64["wall_s"],
            "speedup_fp32_mixed_over_fp64": ps32 / (sc.n * K64 / r64["wall_s"])},
        fp32_mixed_cold_gjk={"particle_steps_per_s": sc.n * K / r32c["wall_s"],
                             "ms_per_step": r32c["wall_s"] * 1e3 / K,
                             "gjk_iterations_cold": r32c["stats"]["gjk_iterations"],
                             "gjk_iterations_warm": st["gjk_iterations"]},
        fp32_mixed_error_vs_fp64=agit,
        fp32_mixed_error_vs_fp64_bed_at_rest=err,
        gjk_pair_tests_per_s=st["gjk_calls"] / 2 / r32["wall_s"],
        gjk_pair_tests_note="unordered pairs that reached GJK (each is visited from both particles)",
        step_stats=step_stats(st),
        phase_ms_per_step=r32["phases"],
        gjk_microbench={"fp64": mb64, "fp32": mb32},
        roofline=roofline,
        roofline_second=roof_other,
        roofline_valu=valu_roofline(r32, K),
        roofline_step_hbm=roofline_step,
        cpu_baseline=cpu)
    if cpu:
        out["speedup_vs_cpu"] = ps32 / cpu["value"]
        out["speedup_vs_cpu_1_thread"] = ps32 / cpu["single_thread"]["value"]
    return out


def bench_c0(args):
    """The reference's CPU-runnable case: 1,000 spheres (r = 0.5 mm) on a
    jittered 10^3 lattice in a 12 mm walled box, Hooke kn = 1e5, en = 0.8,
    mu = 0.3, gravity, dt = 1e-6, 1,000 steps of explicit Euler, FP64 (the
    plain path), every step replayed from one captured graph."""
    K = args.steps or 1000
    W = args.warmup
    sc = S.config0()
    log(f"c0: FP64, {W} warm-up + profiled + {K} timed steps")
    r64 = run_engine(sc, A.FP64, W, K)
    ps = sc.n * K / r64["wall_s"]
    log(f"  {r64['wall_s'] * 1e3 / K:.4f} ms/step, {ps:.3e} particle-steps/s")
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(sc, args.cpu_seconds, "the same 1,000-sphere box")
    st = r64["stats"]
    step_ms = r64["wall_s"] * 1e3 / K
    phases = r64["phases"]
    dom = max(phases, key=phases.get)
    return contract(
        "particle-steps/s (FP64) on the 1,000-sphere box", ps, K, W, step_ms, "f64",
        {"workload": "c0 spheres: 1000 spheres r=0.5 mm on a jittered 10^3 lattice, 12 mm walled box, "
                     "kn=1e5, en=0.8, mu=0.3, dt=1e-6, 1000 steps, FP64",
         "n_particles": sc.n, "precision": "FP64"},
        step_stats=step_stats(st), phase_ms_per_step=phases,
        roofline=dict(bound="hbm", kernel=f"the step (largest phase: {dom})", bytes_per_particle_step=B_PS_FP64,
                      achieved=B_PS_FP64 * ps / 1e9, peak=PEAK_HBM_GBS, unit="GB/s",
                      frac=B_PS_FP64 * ps / 1e9 / PEAK_HBM_GBS, traffic=None,
                      note="1,000 particles fill no device: the step is bound by its ~12 kernel launches "
                           "(replayed from a graph), not by HBM"),
        cpu_baseline=cpu, speedup_vs_cpu=None if cpu is None else ps / cpu["value"],
        speedup_vs_cpu_1_thread=None if cpu is None else ps / cpu["single_thread"]["value"])


def bench_c2(args):
    """Polydisperse polyhedra: 250k cubes, 8-vertex hulls and spheres (size
    ratio 3:1), Gaussian velocities, phi ~0.45, walled, dt = 5e-7, 2000
    steps, FP32-mixed, with FP64 beside it."""
    K = args.steps or 2000
    W = args.warmup
    n = args.n or 250_000
    log(f"generating the polyhedron bed, n = {n}")
    t0 = time.perf_counter()
    sc = S.config2(n=n, log=log)
    log(f"  done in {time.perf_counter() - t0:.1f} s: phi = {sc.notes['phi']:.4f}, rounds = {sc.notes['rounds']}")
    tol = GJK_TOL
    log(f"FP32-mixed: {W} warm-up + profiled + {K} timed steps")
    # ~16 residents per cell on average, up to ~100 where the small grains
    # lie: the half-shell search with its groups from a work list (the
    # automatic choice here)
    r32 = run_engine(sc, A.FP32_MIXED, W, K, flags=FP32_FLAGS, max_neighbors=96)
    ps32 = sc.n * K / r32["wall_s"]
    log(f"  {r32['wall_s'] * 1e3 / K:.3f} ms/step, {ps32:.3e} particle-steps/s")
    r64 = None
    if not args.no_fp64:
        log(f"FP64: {W} warm-up + profiled + {K} timed steps")
        r64 = run_engine(sc, A.FP64, W, K, max_neighbors=96)
        log(f"  {r64['wall_s'] * 1e3 / K:.3f} ms/step")
        g64 = run_engine(sc, A.FP64, W, K, profile=False, gjk_tol=tol[A.FP32_MIXED], max_neighbors=96)
        err = dict(steps=W + K, **pos_error(r32, r64, sc.pos, sc), fp64_at_fp32_gap=pos_error(g64, r64, sc.pos, sc))
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(S.config2(n=8000, seed=7), args.cpu_seconds, "a polyhedron bed of the same distributions")
    st = r32["stats"]
    return contract(
        "particle-steps/s (FP32-mixed) on the polyhedron bed", ps32, K, W, r32["wall_s"] * 1e3 / K, "f32",
        {"workload": "c2 polydisperse polyhedra: 50% cubes, 30% 8-vertex hulls, 20% spheres, size ratio 3:1 "
                     "log-uniform, v~N(0,0.1 m/s), walled, dt=5e-7",
         "n_particles": sc.n, "phi": sc.notes["phi"],
         "precision": "FP32-mixed (FP64 state; FP64 geometry of the pairs in contact)"},
        fp64=None if r64 is None else {
            "particle_steps_per_s": sc.n * K / r64["wall_s"], "ms_per_step": r64["wall_s"] * 1e3 / K,
            "speedup_fp32_mixed_over_fp64": r64["wall_s"] / r32["wall_s"]},
        fp32_mixed_error_vs_fp64=None if r64 is None else err,
        gjk_pair_tests_per_s=st["gjk_calls"] / 2 / r32["wall_s"],
        gjk_iterations_per_test=st["gjk_iterations"] / max(st["gjk_calls"], 1),
        step_stats=step_stats(st), phase_ms_per_step=r32["phases"],
        roofline=integrate_roofline(sc, r32, K), roofline_narrow=narrow_roofline(sc, r32, K),
        roofline_valu=valu_roofline(r32, K), cpu_baseline=cpu,
        speedup_vs_cpu=None if cpu is None else ps32 / cpu["value"])


GRAPH_STEPS_C3 = 100


def bench_c3(args):
    """Batched ensemble: 512 superquadric beds of 500..20,000 particles in one
    context, 100 steps of all of them per launch of one captured graph; cell
    size, block size, narrow-phase residency and pass structure chosen by the
    autotuner on the ensemble itself."""
    from grains3dgpu_amd.autotune import autotune
    from grains3dgpu_amd.engine import Engine
    K = args.steps or 1000
    W = args.warmup
    log("generating the ensemble (512 beds)")
    t0 = time.perf_counter()
    sc = S.config3(log=log)
    log(f"  done in {time.perf_counter() - t0:.1f} s: {sc.n} particles, rounds = {sc.notes['rounds']}")
    t0 = time.perf_counter()
    tuned = autotune(sc, precision=A.FP32_MIXED, flags=FP32_FLAGS, gjk_rel_tol=GJK_TOL[A.FP32_MIXED], steps=10,
                     log=log)
    tune_s = time.perf_counter() - t0
    log(f"  autotuner: {tuned['cell_size_factor']}, {tuned['block_size']}, {tuned['narrow_blocks_per_cu']}, "
        f"{tuned['narrow_passes']} in {tune_s:.1f} s")
    launch = dict(block_size=tuned["block_size"], narrow_blocks_per_cu=tuned["narrow_blocks_per_cu"],
                  narrow_passes=tuned["narrow_passes"], candidate_staging=tuned["candidate_staging"])
    # 100 steps of all 512 beds per graph launch
    r32 = run_engine(sc, A.FP32_MIXED, W, K, flags=FP32_FLAGS, graph_steps=GRAPH_STEPS_C3, **launch)
    ps32 = sc.n * K / r32["wall_s"]
    log(f"  {r32['wall_s'] * 1e3 / K:.3f} ms/step, {ps32:.3e} particle-steps/s ({GRAPH_STEPS_C3} steps per graph)")
    # one step per graph launch, and the untuned default launch, beside it
    o32 = run_engine(sc, A.FP32_MIXED, W, min(K, 200), profile=False, flags=FP32_FLAGS, **launch)
    log(f"  one step per graph: {o32['wall_s'] * 1e3 / min(K, 200):.3f} ms/step")
    d32 = run_engine(sc, A.FP32_MIXED, W, min(K, 200), profile=False, flags=FP32_FLAGS)
    # error of the tuned FP32-mixed run against FP64 after a fixed 1,000 steps
    err = None
    if not args.no_fp64:
        log("errors after 1,000 steps: FP32-mixed (tuned launch) and FP64")
        e32 = run_engine(sc, A.FP32_MIXED, 0, 1000, profile=False, flags=FP32_FLAGS, **launch)
        e64 = run_engine(sc, A.FP64, 0, 1000, profile=False)
        err = dict(steps=1000, contacts_fp64=e64["stats"]["contacts"], contacts_fp32=e32["stats"]["contacts"],
                   fp64_particle_steps_per_s=sc.n * 1000 / e64["wall_s"], **pos_error(e32, e64, sc.pos, sc))
    cpu = None
    if not args.no_cpu:
        k = int(np.argmin(np.abs(np.array(sc.notes["sizes"]) - 5000)))
        one = S.config3(n_sims=1, n_range=(sc.notes["sizes"][k], sc.notes["sizes"][k] + 1), seed=3 + k)
        cpu = cpu_baseline(one, args.cpu_seconds, "one bed of the ensemble's distribution")
    del Engine
    return contract(
        "particle-steps/s (FP32-mixed) of the batched ensemble", ps32, K, W, r32["wall_s"] * 1e3 / K, "f32",
        {"workload": "c3 ensemble: 512 superquadric beds, sizes log-uniform in [500, 20000], kn~U[5e4,5e5], "
                     "mu~U[0.1,0.5], each its own seed, one context, 100 steps per graph launch",
         "n_particles": sc.n, "n_sims": len(sc.sims),
         "precision": "FP32-mixed (FP64 state; FP64 geometry of the pairs in contact)"},
        autotune=dict(tuned, seconds=tune_s),
        graph_steps=GRAPH_STEPS_C3,
        one_step_graph_particle_steps_per_s=sc.n * min(K, 200) / o32["wall_s"],
        default_launch_particle_steps_per_s=sc.n * min(K, 200) / d32["wall_s"],
        fp32_mixed_error_vs_fp64=err,
        step_stats=step_stats(r32["stats"]), phase_ms_per_step=r32["phases"],
        gjk_pair_tests_per_s=r32["stats"]["gjk_calls"] / 2 / r32["wall_s"],
        roofline=integrate_roofline(sc, r32, K),
        roofline_narrow=narrow_roofline(sc, r32, K), roofline_valu=valu_roofline(r32, K), cpu_baseline=cpu,
        speedup_vs_cpu=None if cpu is None else ps32 / cpu["value"])


def bench_c4(args):
    """Differentiable calibration: 8,192 spheres and ellipsoids settle for
    2,000 steps; loss = relative squared errors of the bed height and mean
    kinetic energy against a target run (kn = 2e5, e = 0.7, mu = 0.4);
    gradients with respect to (kn, e, mu) of each of the three contact-table
    entries through the adjoint (checkpoints every 100 steps), against
    central finite differences, in FP64 and FP32-mixed."""
    import torch
    from grains3dgpu_amd import adjoint
    from grains3dgpu_amd.engine import Engine
    K = args.steps or 2000
    n = args.n or 8192
    every = 100
    log(f"generating the calibration bed, n = {n}")
    sc = S.config4(n=n, log=log)
    mass = adjoint.masses(sc)
    p0 = np.array(sc.tables)[:, [0, 1, 3]].copy()
    pt = np.tile([2e5, 0.7, 0.4], (p0.shape[0], 1))
    res = {}
    for prec, name in ((A.FP64, "fp64"), (A.FP32_MIXED, "fp32_mixed")):
        e = S.load(Engine(dt=sc.dt, precision=prec, gjk_rel_tol=GJK_TOL[prec]), sc)

        def final(params):
            s2 = adjoint.with_params(sc, params)
            e.set_contact_tables(s2)
            e.set_state(s2.pos, s2.quat, s2.vel, s2.omega)
            e.step(K, graph=True)
            p, _, v, _ = e.get_state()
            return p, v

        def loss_of(p, v, target):
            return adjoint.bed_loss(torch.from_numpy(p), torch.from_numpy(v), torch.from_numpy(mass), target)[0].item()

        pT, vT = final(pt)
        target = (float(pT[:, 2].mean()), float((0.5 * mass * (vT * vT).sum(1)).mean()))
        t0 = time.perf_counter()
        final(p0)
        fwd_plain = time.perf_counter() - t0
        params = torch.tensor(p0, requires_grad=True)
        t0 = time.perf_counter()
        pos, quat, vel, om = adjoint.simulate(e, sc, params, K, every)
        fwd = time.perf_counter() - t0
        L, h, ke = adjoint.bed_loss(pos, vel, torch.from_numpy(mass), target)
        t0 = time.perf_counter()
        L.backward()
        bwd = time.perf_counter() - t0
        g = params.grad.numpy().copy()
        # central differences of the loss at several relative steps: below
        # ~1e-4 the GJK witness noise of curved contacts (it converges like
        # the square root of the gap) dominates, above ~1e-2 contact
        # events inside the step; the FP32-mixed forward carries FP32
        # rounding in every force, so its differences are taken at 1e-3 only
        fds = {}
        for rel in ((1e-3, 1e-4, 1e-5, 1e-6) if prec == A.FP64 else (1e-3,)):
            fd = np.zeros_like(p0)
            for r in range(p0.shape[0]):
                for c in range(3):
                    hstep = rel * p0[r, c]
                    pp, pm = p0.copy(), p0.copy()
                    pp[r, c] += hstep
                    pm[r, c] -= hstep
                    fd[r, c] = (loss_of(*final(pp), target) - loss_of(*final(pm), target)) / (2 * hstep)
            fds[rel] = fd
            log(f"  {name}: FD {rel:g} done")
        # errors of sensitivities to relative changes (dL / dlog p: kn in N/m
        # and the dimensionless en, mu on one scale), relative to each
        # entry's largest
        scale = np.abs(g * p0).max(axis=1, keepdims=True)
        errs = {rel: np.abs(g - fd) * p0 / scale for rel, fd in fds.items()}
        best = np.min(np.stack(list(errs.values())), axis=0)
        # a component's difference is trusted where two adjacent steps agree
        # to 1e-3 of that scale (no contact event or noise inside either
        # step); the adjoint against those references
        rels = sorted(fds, reverse=True)
        trusted, terr = 0, 0.0
        for r in range(p0.shape[0]):
            for c in range(3):
                for a, b in zip(rels, rels[1:]):
                    fa, fb = fds[a][r, c] * p0[r, c], fds[b][r, c] * p0[r, c]
                    if abs(fa - fb) <= 1e-3 * scale[r, 0]:
                        trusted += 1
                        terr = max(terr, abs(g[r, c] * p0[r, c] - 0.5 * (fa + fb)) / scale[r, 0])
                        break
        res[name] = dict(
            loss=float(L), bed_height=float(h), mean_ke=float(ke), target=target, grad=g.tolist(),
            fd={f"{rel:g}": fd.tolist() for rel, fd in fds.items()},
            rel_err_vs_fd={f"{rel:g}": float(er.max()) for rel, er in errs.items()},
            rel_err_vs_fd_best_step=float(best.max()),
            fd_trusted_components=f"{trusted} of {g.size}", rel_err_vs_trusted_fd=terr,
            fd_spread=float((np.ptp(np.stack(list(fds.values())), axis=0) * p0 / scale).max()),
            error_note="errors of dL/dlog p per contact-table entry, relative to the entry's largest",
            forward_ms_per_step=fwd_plain * 1e3 / K, recorded_forward_ms_per_step=fwd * 1e3 / K,
            adjoint_ms_per_step=bwd * 1e3 / K, contacts=e.get_stats()["contacts"])
        log(f"  {name}: loss {float(L):.4e}, grad {g.tolist()}, fd(1e-3) {fds[1e-3].tolist()}")
        e.close()
    g64, g32 = np.array(res["fp64"]["grad"]), np.array(res["fp32_mixed"]["grad"])
    sc64 = np.abs(g64 * p0).max(1, keepdims=True)
    res["fp32_mixed"]["grad_rel_diff_vs_fp64"] = float((np.abs(g32 - g64) * p0 / sc64).max())
    res["fp32_mixed"]["rel_err_vs_fp64_fd_1e-3"] = float(
        (np.abs(g32 - np.array(res["fp64"]["fd"]["0.001"])) * p0 / sc64).max())
    r = res["fp64"]
    total = (r["recorded_forward_ms_per_step"] + r["adjoint_ms_per_step"]) * 1e-3 * K
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(sc, args.cpu_seconds, "the same bed, forward only (the oracle has no adjoint)")
    return contract(
        "particle-steps/s of forward + adjoint sweep (FP64) on the calibration bed", n * K / total, K, 0,
        total * 1e3 / K, "f64",
        {"workload": "c4 calibration: 8192 spheres + ellipsoids (ratio <= 2:1), phi=0.35, walled, "
                     "2000 steps at dt=1e-6, checkpoints every 100, gradients wrt kn, e, mu of 3 table entries",
         "n_particles": n, "checkpoint_every": every},
        fp64=res["fp64"], fp32_mixed=res["fp32_mixed"], roofline=None, cpu_baseline=cpu)


def main():
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=None, help="timed steps (default: the workload's)")
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--n", type=int, default=None, help="particles (default: the workload's)")
    ap.add_argument("--workload", default="c1", choices=("c0", "c1", "c2", "c3", "c4"),
                    help="c1 superquadric bed (default), c0 1,000-sphere box, c2 polyhedra, c3 batched ensemble, "
                         "c4 adjoint")
    ap.add_argument("--fp64-steps", type=int, default=200)
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fp64", action="store_true")
    ap.add_argument("--eager", action="store_true",
                    help="launch the timed steps one kernel at a time instead of replaying a captured graph "
                         "(profiler runs: kernel times are the same)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only copy 1 GiB device to device three times (reference for the HBM byte counters)")
    args = ap.parse_args()
    if args.copy_calibration:
        copy_calibration()
        return
    if args.eager:
        global EAGER
        EAGER = True
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {args.gpus}); "
              "the batched multi-simulation form is the way to fill one device", file=sys.stderr)
        sys.exit(2)
    out = {"c0": bench_c0, "c1": bench_c1, "c2": bench_c2, "c3": bench_c3, "c4": bench_c4}[args.workload](args)
    out["timed_steps_launch"] = "eager" if EAGER else "graph"
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
