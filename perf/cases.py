"""Cases of the framework's main path: time steps of particle beds (every shape family, both precisions, both
semantics, one and many simulations), the driver's step-by-step loop, the calibration's forward run and reverse
sweep, and the batched GJK distances -- each through the entry points a program calls (grains3dgpu_amd.engine,
grains3dgpu_amd.adjoint).

A stepping pass is a restart from a checkpoint: restore the state, run the steps, read the state back.  It takes
the same steps every time, so passes on one state are alike.
"""
import ctypes
import math

import numpy as np
import torch

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import adjoint
from grains3dgpu_amd import scene as S
from grains3dgpu_amd.engine import Engine

# the FP32-mixed form of long runs: warm-started searches, FP64 geometry of the pairs in contact
MIXED = A.WARM_START | A.FP64_CONTACTS
TOL = {A.FP64: 1e-10, A.FP32_MIXED: 1e-6}


def listed():
    return [
        # the smallest run: the walled box of 1,000 spheres, launch-bound
        dict(name="spheres_1000", form="spheres", n=1000, steps=100, fp64=True, quirks=False),
        # a driver that calls the component manager once per step and reads the contact counts (C++ loop of the
        # reference's main program), on a small box with the reference semantics
        dict(name="driver_343", form="driver", n=343, steps=20, fp64=True, quirks=True),
        # the headline workload: a large bed of superquadrics at rest between a floor and a ceiling
        dict(name="superquadrics_1m", form="loose", n=1_000_000, steps=200, fp64=False, agitated=False),
        # an agitated bed of ordinary size, odd count
        dict(name="superquadrics_50k", form="loose", n=50_653, steps=200, fp64=False, agitated=True),
        # a touching packing in plain FP64: the accuracy runs of the beds
        dict(name="packing_fp64_8k", form="packed", n=8_191, steps=40, fp64=True, agitated=True),
        # the same kind of packing in the mixed form: every grain in contact
        dict(name="packing_mixed_30k", form="packed", n=29_791, steps=100, fp64=False, agitated=True),
        # polydisperse cubes, hulls and spheres in a walled box: dense cells
        dict(name="polyhedra_100k", form="polyhedra", n=100_003, steps=100, fp64=False),
        # many independent beds in one context, many steps per captured graph
        dict(name="ensemble_64", form="ensemble", n=64, lo=500, hi=20_000, steps=50, fp64=False),
        # calibration: forward run and reverse sweep of spheres and ellipsoids in FP64
        dict(name="calibration_4096", form="calibration", n=4096, steps=40, fp64=True),
        # the reference's narrow phase (Johnson's sub-algorithm) on boxes and superquadrics
        dict(name="reference_4k", form="reference", n=4_001, steps=40, fp64=True),
        # cylinders and cones with rolling resistance, a Box obstacle, leapfrog; cold starts
        dict(name="cylinders_cones_3k", form="cylcone", n=3_001, steps=100, fp64=False),
        # the reference's GJK microbenchmark on device buffers
        dict(name="gjk_614400", form="gjk", n=614_400, fp64=False, quirks=True),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["spheres", "driver", "loose", "loose", "packed", "packed", "polyhedra", "ensemble",
                       "calibration", "reference", "cylcone", "gjk"])
    fp64 = rng.random() < 0.5
    if form == "spheres":
        return dict(form=form, n=_logu(rng, 200, 200_000), steps=rng.randint(20, 120), fp64=fp64,
                    quirks=rng.random() < 0.3)
    if form == "driver":
        return dict(form=form, n=_logu(rng, 60, 5_000), steps=rng.randint(5, 30), fp64=True, quirks=rng.random() < 0.5)
    if form == "loose":
        n = _logu(rng, 2_000, 300_000 if fp64 else 1_000_000)
        return dict(form=form, n=n, steps=rng.randint(10, 40 if fp64 else 150), fp64=fp64, agitated=rng.random() < 0.5)
    if form == "packed":
        return dict(form=form, n=_logu(rng, 500, 15_000 if fp64 else 100_000), steps=rng.randint(20, 60), fp64=fp64,
                    agitated=rng.random() < 0.5)
    if form == "polyhedra":
        return dict(form=form, n=_logu(rng, 3_000, 150_000), steps=rng.randint(20, 100), fp64=fp64)
    if form == "ensemble":
        lo = _logu(rng, 300, 1_000)
        return dict(form=form, n=rng.randint(3, 80), lo=lo, hi=lo * rng.randint(2, 20), steps=rng.randint(20, 50),
                    fp64=False)
    if form == "calibration":
        return dict(form=form, n=_logu(rng, 256, 8_192), steps=rng.randint(10, 40), fp64=True)
    if form == "reference":
        return dict(form=form, n=_logu(rng, 300, 8_000), steps=rng.randint(10, 40), fp64=True)
    if form == "cylcone":
        return dict(form=form, n=_logu(rng, 500, 20_000), steps=rng.randint(20, 100), fp64=fp64)
    return dict(form=form, n=_logu(rng, 1_000, 600_000), fp64=fp64, quirks=rng.random() < 0.5)


# ---- scenes ---------------------------------------------------------------------------------------------------
def _lattice(n):
    side = int(math.ceil(n ** (1.0 / 3.0) - 1e-9))
    idx = np.arange(n)
    cz, rem = np.divmod(idx, side * side)
    cy, cx = np.divmod(rem, side)
    return side, int(cz[-1]) + 1, np.stack([cx, cy, cz], 1)


def _walled(lo, hi, first):
    """Six walls of the box [lo, hi] as shape records, their shape ids and poses."""
    ws, tr = S.box_walls(lo, hi)
    rec = S.shape_records(A.RECTANGLE, [w["dims"] for w in ws], 0.0, 0.0)
    return rec, np.arange(first, first + 6, dtype=np.uint32), tr


def _floor_ceiling(L, z0, first):
    rec = S.shape_records(A.RECTANGLE, [[0.5 * L[0], 0.5 * L[1]]] * 2, 0.0, 0.0)
    eye = [1, 0, 0, 0, 1, 0, 0, 0, 1.0]
    tr = np.array([eye + [0.5 * L[0], 0.5 * L[1], z0], eye + [0.5 * L[0], 0.5 * L[1], L[2]]])
    return rec, np.array([first, first + 1], np.uint32), tr


def _spheres(n, seed):
    """Spheres (r = 0.5 mm) on a jittered cubic lattice whose neighbours overlap by about 1 %, in a walled box."""
    rng = np.random.default_rng(seed)
    side, layers, c = _lattice(n)
    sp = 0.99e-3
    pos = (c + 0.5) * sp + rng.uniform(-0.02e-3, 0.02e-3, (n, 3))
    hi = (side * sp, side * sp, layers * sp)
    wall, osh, otr = _walled((0, 0, 0), hi, 1)
    return S.Scene(shapes=np.concatenate([S.shape_records(A.SPHERE, [[0.5e-3]], 2.5e-5, 2500.0), wall]),
                   tables=np.array([S.hooke_row(1e5, 0.8, 2e4, 0.3)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=hi, gravity=(0, 0, -9.81))],
                   particle_shape=np.zeros(n, np.uint32), pos=pos, quat=S.random_quaternions(rng, n),
                   vel=rng.normal(0, 0.02, (n, 3)), omega=rng.normal(0, 20.0, (n, 3)), obstacle_shape=osh,
                   obstacle_tr=otr, dt=1e-7)


TILE = 32 ** 3


def _loose_bed(rng, n, a_rng, half):
    """n superquadrics of random axes, blockiness and orientation, each inside its own box of a cubic lattice
    (half-side `half`): orientations redrawn while one sticks out, what still does scaled down; then moved at
    random within its box.  Large beds repeat a tile of grains (moved differently)."""
    m = min(n, TILE)
    prm = S.superquadric_params(rng, m, a_rng=a_rng)
    quat = S.random_quaternions(rng, m)
    ext = np.stack([S.superquadric_extent(prm, quat, k) for k in range(3)], 1)
    for _ in range(3):
        bad = np.flatnonzero(ext.max(1) > half)
        quat[bad] = S.random_quaternions(rng, len(bad))
        ext[bad] = np.stack([S.superquadric_extent(prm[bad], quat[bad], k) for k in range(3)], 1)
    f = np.minimum(1.0, 0.999 * half / ext.max(1))
    prm[:, :3] *= f[:, None]
    ext *= f[:, None]
    k = np.arange(n) % m
    side, layers, c = _lattice(n)
    pos = (c + 0.5) * (2 * half) + rng.uniform(-1, 1, (n, 3)) * 0.95 * (half - ext[k])
    return prm[k], pos, quat[k], (2 * half * side, 2 * half * side, 2 * half * layers)


def _loose(n, seed, agitated):
    """Superquadrics, a, b, c in [0.4, 1] mm, n1, n2 in [2, 8], solid fraction about 0.3, periodic in x and y
    between a floor and a ceiling; at rest, or agitated."""
    rng = np.random.default_rng(seed)
    prm, pos, quat, L = _loose_bed(rng, n, (0.4e-3, 1e-3), 0.95e-3)
    wall, osh, otr = _floor_ceiling(L, 0.0, n)
    etat = S.matched_etat(1e5, 0.8, 2.5e-6)
    return S.Scene(shapes=np.concatenate([S.shape_records(A.SUPERQUADRIC, prm, 0.05 * prm[:, :3].min(1), 2500.0), wall]),
                   tables=np.array([S.hooke_row(1e5, 0.8, etat, 0.3)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=L, gravity=(0, 0, -9.81), periodic=0b011)],
                   particle_shape=np.arange(n, dtype=np.uint32), pos=pos, quat=quat,
                   vel=rng.normal(0, 0.2, (n, 3)) * agitated, omega=rng.normal(0, 100.0, (n, 3)) * agitated,
                   obstacle_shape=osh, obstacle_tr=otr, dt=1e-6)


def _packed(n, seed, agitated):
    """Superquadrics of semi-axes 2.5 mm and random blockiness, tilted by at most 0.05 rad, on a lattice whose
    neighbours' crusts overlap: contacts on every side of every grain."""
    rng = np.random.default_rng(seed)
    a, ct = 2.5e-3, 0.25e-3
    sp = 2 * a - 0.2 * ct
    side, layers, c = _lattice(n)
    prm = np.concatenate([np.full((n, 3), a), rng.uniform(2, 8, (n, 2))], 1)
    ax = rng.standard_normal((n, 3))
    ax /= np.linalg.norm(ax, axis=1, keepdims=True)
    ang = rng.uniform(0, 0.05, n)
    quat = np.concatenate([ax * np.sin(ang / 2)[:, None], np.cos(ang / 2)[:, None]], 1)
    hi = (side * sp, side * sp, layers * sp)
    wall, osh, otr = _walled((0, 0, 0), hi, n)
    return S.Scene(shapes=np.concatenate([S.shape_records(A.SUPERQUADRIC, prm, ct, 2500.0), wall]),
                   tables=np.array([S.hooke_row(1e5, 0.8, 2e3, 0.3)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=hi, gravity=(0, 0, -9.81))],
                   particle_shape=np.arange(n, dtype=np.uint32), pos=(c + 0.5) * sp, quat=quat,
                   vel=rng.normal(0, 0.05, (n, 3)) * agitated, omega=rng.normal(0, 20.0, (n, 3)) * agitated,
                   obstacle_shape=osh, obstacle_tr=otr, dt=1e-6)


def _ensemble(n_sims, lo, hi, seed):
    """n_sims independent beds (as _loose, sizes log-uniform in [lo, hi]), each with its own stiffness and
    friction, in one context."""
    rng = np.random.default_rng(seed)
    sizes = np.exp(np.random.default_rng(5 + n_sims).uniform(math.log(lo), math.log(hi), n_sims)).astype(int)
    beds = [_loose_bed(rng, int(m), (0.4e-3, 1e-3), 0.95e-3) for m in sizes]
    n = int(sizes.sum())
    prm = np.concatenate([b[0] for b in beds])
    kn, mu = rng.uniform(5e4, 5e5, n_sims), rng.uniform(0.1, 0.5, n_sims)
    walls, osh, otr = zip(*[_floor_ceiling(b[3], 0.0, n + 2 * k) for k, b in enumerate(beds)])
    return S.Scene(shapes=np.concatenate([S.shape_records(A.SUPERQUADRIC, prm, 0.05 * prm[:, :3].min(1), 2500.0), *walls]),
                   tables=np.array([S.hooke_row(kn[k], 0.8, S.matched_etat(kn[k], 0.8, 2.5e-6), mu[k])
                                    for k in range(n_sims)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=b[3], gravity=(0, 0, -9.81), periodic=0b011,
                              contact_table=k) for k, b in enumerate(beds)],
                   particle_shape=np.arange(n, dtype=np.uint32), particle_sim=np.repeat(np.arange(n_sims), sizes).astype(np.uint32),
                   pos=np.concatenate([b[1] for b in beds]), quat=np.concatenate([b[2] for b in beds]),
                   vel=rng.normal(0, 0.1, (n, 3)), omega=rng.normal(0, 50.0, (n, 3)),
                   obstacle_shape=np.concatenate(osh), obstacle_sim=np.repeat(np.arange(n_sims), 2).astype(np.uint32),
                   obstacle_tr=np.concatenate(otr), dt=1e-6)


def _reference(n, seed):
    """Boxes and superquadrics (half extents about 2.5 mm), nearly aligned on a lattice that leaves gaps and small
    overlaps, in a walled box, for the reference semantics."""
    rng = np.random.default_rng(seed)
    side, layers, c = _lattice(n)
    a, sp = 2.5e-3, 5.02e-3
    prm = np.concatenate([rng.uniform(0.96, 1.0, (n, 3)) * a, rng.uniform(2, 8, (n, 2))], 1)
    box = rng.uniform(size=n) < 0.5
    rec = S.shape_records(A.SUPERQUADRIC, prm, 0.05 * a, 2500.0)
    rec["kind"][box] = A.BOX
    rec["dims"][box, 3:] = 0.0
    ax = rng.standard_normal((n, 3))
    ax /= np.linalg.norm(ax, axis=1, keepdims=True)
    ang = rng.uniform(0, 0.1, n)
    quat = np.concatenate([ax * np.sin(ang / 2)[:, None], np.cos(ang / 2)[:, None]], 1)
    hi = (side * sp, side * sp, layers * sp)
    wall, osh, otr = _walled((0, 0, 0), hi, n)
    return S.Scene(shapes=np.concatenate([rec, wall]), tables=np.array([S.hooke_row(1e5, 0.8, 2e3, 0.3)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=hi, gravity=(0, 0, -9.81))],
                   particle_shape=np.arange(n, dtype=np.uint32), pos=(c + 0.5) * sp, quat=quat,
                   vel=rng.normal(0, 0.05, (n, 3)), omega=rng.normal(0, 5.0, (n, 3)), obstacle_shape=osh,
                   obstacle_tr=otr, dt=1e-6)


def _cylcone(n, seed):
    """Upright cylinders and cones (r = 2.25 mm, h = 5 mm, axis turned onto z, tilted by at most 0.05 rad) in
    columns whose crusts overlap, rolling resistance on, periodic in x and y between a floor and a ceiling; a Box
    obstacle stands in the middle, over the columns it replaces."""
    rng = np.random.default_rng(seed)
    r, h = 2.25e-3, 5e-3
    ct = 0.1 * r
    sx, sz = 2 * r - 0.2 * ct, h - 0.2 * ct
    side = max(8, int(math.ceil(n ** (1.0 / 3.0))))
    free = np.array([(i, j) for j in range(side) for i in range(side)
                     if not (abs(i - side // 2) <= 0 and abs(j - side // 2) <= 0)])
    k = np.arange(n)
    layer, col = np.divmod(k, len(free))
    ij = free[col]
    cone = (ij.sum(1) % 2).astype(np.uint32)
    z0 = np.where(cone == 1, 0.25 * h, 0.5 * h) + r * math.sin(0.05)
    pos = np.stack([(ij[:, 0] + 0.5) * sx, (ij[:, 1] + 0.5) * sx, z0 + layer * sz], 1)
    s = math.sin(math.pi / 4)
    ax = rng.standard_normal((n, 3))
    ax /= np.linalg.norm(ax, axis=1, keepdims=True)
    ang = rng.uniform(0, 0.05, n)
    t = np.concatenate([ax * np.sin(ang / 2)[:, None], np.cos(ang / 2)[:, None]], 1)
    quat = s * np.stack([t[:, 3] + t[:, 0], t[:, 1] + t[:, 2], t[:, 2] - t[:, 1], t[:, 3] - t[:, 0]], 1)
    L = (side * sx, side * sx, (layer[-1] + 1) * sz + h)
    wall, osh, otr = _floor_ceiling(L, 0.0, 3)
    b = 0.95 * 0.5 * sx
    mid = (side // 2 + 0.5) * sx
    rec = np.concatenate([S.shape_records(A.CYLINDER, [[r, h]], ct, 2500.0), S.shape_records(A.CONE, [[r, h]], ct, 2500.0),
                          S.shape_records(A.BOX, [[b, b, 0.5 * L[2]]], 0.05 * b, 0.0), wall])
    return S.Scene(shapes=rec, tables=np.array([S.hooke_row(1e5, 0.8, 2e3, 0.3, 1e-6)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=L, gravity=(0, 0, -9.81), periodic=0b011)],
                   particle_shape=cone, pos=pos, quat=quat, vel=rng.normal(0, 0.05, (n, 3)),
                   omega=rng.normal(0, 5.0, (n, 3)), obstacle_shape=np.concatenate([osh, [2]]).astype(np.uint32),
                   obstacle_tr=np.concatenate([otr, [[1, 0, 0, 0, 1, 0, 0, 0, 1.0, mid, mid, 0.5 * L[2]]]]), dt=1e-6)


def _pairs(n, seed):
    """The reference's GJK microbenchmark pairs: centres N(-0.05, 0.005) and N(0.05, 0.005) per axis, uniform
    orientations."""
    rng = np.random.default_rng(seed)
    return [S.transform12(rng.normal(s * 0.05, 0.005, (n, 3)), S.random_quaternions(rng, n)) for s in (-1, 1)]


def _scene(case, seed):
    f, n = case["form"], case["n"]
    if f in ("spheres", "driver"):
        return _spheres(n, seed)
    if f == "loose":
        return _loose(n, seed, case["agitated"])
    if f == "packed":
        return _packed(n, seed, case["agitated"])
    if f == "polyhedra":
        return S.config2(n=n, seed=seed, phi=0.47, resolve=False)
    if f == "ensemble":
        return _ensemble(n, case["lo"], case["hi"], seed)
    if f == "calibration":
        return S.config4(n=n, seed=seed, resolve=False)
    if f == "reference":
        return _reference(n, seed)
    return _cylcone(n, seed)


# ---- one pass -------------------------------------------------------------------------------------------------
def prepare(case, seed):
    form = case["form"]
    prec = A.FP64 if case["fp64"] else A.FP32_MIXED
    if form == "gjk":
        e = Engine(precision=prec, flags=A.REF_QUIRKS if case["quirks"] else 0)
        one = _spheres(1, 0)
        one.shapes = [dict(kind=A.SUPERQUADRIC, dims=(0.05, 0.05, 0.05, 3.0, 3.0), density=1.0)]
        e.set_shapes(one)
        n = case["n"]
        ta, tb = (torch.from_numpy(t).cuda() for t in _pairs(n, seed))
        z = torch.zeros(n, dtype=torch.int32, device="cuda")
        return dict(case=case, engine=e, z=z, ta=ta, tb=tb, dist=torch.empty(n, dtype=torch.float64, device="cuda"),
                    iters=torch.empty(n, dtype=torch.int32, device="cuda"))
    sc = _scene(case, seed)
    flags = 0
    if form == "reference" or case.get("quirks"):
        flags = A.REF_QUIRKS
    elif form not in ("cylcone", "calibration") and not case["fp64"]:
        flags = MIXED
    e = Engine(dt=sc.dt, precision=prec, flags=flags, gjk_rel_tol=0.0 if flags == A.REF_QUIRKS else TOL[prec],
               max_neighbors=96 if form == "polyhedra" else 64,
               integrator=A.SECOND_ORDER_LEAPFROG if form == "cylcone" else A.FIRST_ORDER_EXPLICIT)
    S.load(e, sc)
    if form == "ensemble":
        e.set_graph_steps(case["steps"])
    st = dict(case=case, engine=e)
    if form == "calibration":
        st.update(scene=sc, params=torch.tensor(np.array(sc.tables)[:, [0, 1, 3]]),
                  mass=torch.from_numpy(adjoint.masses(sc)))
    else:
        st["checkpoint"] = e.snapshot()
    return st


def run(state):
    case, e = state["case"], state["engine"]
    form = case["form"]
    if form == "gjk":
        ms = ctypes.c_float()
        e._chk(e.L.grains_gjk_batch_device(e.h, state["z"].data_ptr(), state["z"].data_ptr(), state["ta"].data_ptr(),
                                           state["tb"].data_ptr(), case["n"], state["dist"].data_ptr(),
                                           state["iters"].data_ptr(), ctypes.byref(ms)))
        return {"dist": state["dist"], "iters": state["iters"]}
    if form == "calibration":
        p = state["params"].clone().requires_grad_(True)
        pos, quat, vel, omega = adjoint.simulate(e, state["scene"], p, case["steps"], checkpoint_every=20)
        loss, _, _ = adjoint.bed_loss(pos, vel, state["mass"], (0.03, 1e-6))
        loss.backward()
        return {"pos": pos.detach(), "quat": quat.detach(), "vel": vel.detach(), "omega": omega.detach(), "grad": p.grad}
    e.restore(state["checkpoint"])
    if form == "driver":
        for _ in range(case["steps"]):
            e.step(1)
            contacts = e.get_contact_count()
        force, torque = e.get_torce()
    else:
        e.step(case["steps"], graph=True)
        contacts = e.get_contact_count()
    pos, quat, vel, omega = e.get_state()
    out = {"pos": pos, "quat": quat, "vel": vel, "omega": omega, "contacts": contacts}
    if form == "driver":
        out.update(force=force, torque=torque)
    return out


def _particles(case):
    if case["form"] != "ensemble":
        return case["n"]
    rng = np.random.default_rng(5 + case["n"])
    return int(np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["n"])).astype(int).sum())


def work(case):
    """Per particle and step: the state (13 doubles) read and written, its shape's record and mass properties read
    (200 B); about 100 operations to move it and 40 (spheres) or 400 (GJK) for each of six neighbours.  The reverse
    sweep runs every step twice more and differentiates it.  Per GJK pair: two transforms read, distance and
    iterations written, eight iterations of 220 operations."""
    n = _particles(case)
    if case["form"] == "gjk":
        return {"bytes": n * (2 * 96 + 2 * 4 + 12), "flops": n * 8 * 220}
    k = case["steps"] * (4 if case["form"] == "calibration" else 1)
    per = 40 if case["form"] in ("spheres", "driver") else 400
    return {"bytes": n * k * (2 * 104 + 200), "flops": n * k * (100 + 6 * per)}


# ---- the sphere cases in plain numpy ----------------------------------------------------------------------------
def _neighbours(pos, reach):
    """Pairs i < j closer than reach, by cells of that side."""
    c = np.floor(pos / reach).astype(np.int64) + 1
    w = c.max(0) + 2
    key = (c[:, 2] * w[1] + c[:, 1]) * w[0] + c[:, 0]
    order = np.argsort(key, kind="stable")
    ks = key[order]
    out = []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                k = key + (dz * w[1] + dy) * w[0] + dx
                a, b = np.searchsorted(ks, k), np.searchsorted(ks, k, side="right")
                for s in range(int((b - a).max(initial=0))):
                    i = np.flatnonzero(a + s < b)
                    out.append(np.stack([i, order[a[i] + s]], 1))
    p = np.concatenate(out)
    p = p[p[:, 0] < p[:, 1]]
    return p[np.linalg.norm(pos[p[:, 1]] - pos[p[:, 0]], axis=1) < reach]


def _snap(v):
    return np.where(np.abs(v) < 1e-10, 0.0, v)


def _hooke(row, cv, rel_vel, avmass, omega0, lever):
    """Spring, dashpot, tangential dashpot and Coulomb cap; force on the first body and its moment."""
    kn, en, etat, muc, _ = row
    le = math.log(en)
    damp = -omega0 * le / math.sqrt(math.pi ** 2 + le * le)
    n = _snap(cv / np.linalg.norm(cv, axis=1, keepdims=True))
    vn = (rel_vel * n).sum(1, keepdims=True) * n
    vt = rel_vel - vn
    nvt = np.linalg.norm(vt, axis=1, keepdims=True)
    fn = kn * cv - 2 * damp * avmass * vn
    ft = -2 * etat * avmass * vt
    cap = muc * np.linalg.norm(fn, axis=1, keepdims=True)
    tangent = np.where(nvt > 1e-10, vt / np.maximum(nvt, 1e-300), 0.0)
    f = fn + np.where(cap < np.linalg.norm(ft, axis=1, keepdims=True), -cap * tangent, ft)
    return f, np.cross(lever, f)


def _qmul(a, b):
    v = np.cross(a[:, :3], b[:, :3]) + a[:, 3:] * b[:, :3] + b[:, 3:] * a[:, :3]
    return np.concatenate([v, (a[:, 3] * b[:, 3] - (a[:, :3] * b[:, :3]).sum(1))[:, None]], 1)


def exact(case, seed):
    if case["form"] not in ("spheres", "driver") or not case["fp64"] or case["n"] * case["steps"] > 600_000:
        return None
    sc = _spheres(case["n"], seed)
    x, q, v, w = (np.array(a, np.float64) for a in (sc.pos, sc.quat, sc.vel, sc.omega))
    r, rho, row, dt = 0.5e-3, 2500.0, sc.tables[0], sc.dt
    m = rho * 4.0 * math.pi * r ** 3 / 3.0
    inertia = rho * 8.0 * math.pi / 15.0 * r ** 5
    pairs = _neighbours(x, 2.2 * r)
    i, j = pairs.T
    count = np.zeros(len(x), np.int64)
    for _ in range(case["steps"]):
        F, M = np.zeros_like(x), np.zeros_like(x)
        d = x[j] - x[i]
        dist = np.linalg.norm(d, axis=1)
        over = dist - r - r
        k = np.flatnonzero(over < 0)
        a, b, o, u = i[k], j[k], over[k, None], d[k] / dist[k, None]
        cp = x[a] + (r + 0.5 * o) * u
        # the reference semantics take the contact point in the world as the lever of the relative velocity
        la, lb = (cp, cp) if case["quirks"] else (cp - x[a], cp - x[b])
        rel = (v[a] + np.cross(w[a], la)) - (v[b] + np.cross(w[b], lb))
        f, t = _hooke(row, o * u, rel, 0.5 * m, math.sqrt(row[0] / (0.5 * m)), cp - x[a])
        np.add.at(F, a, f)
        np.add.at(F, b, -f)
        np.add.at(M, a, t)
        np.add.at(M, b, np.cross(cp - x[b], -f))
        count += np.bincount(np.concatenate([a, b]), minlength=len(x))
        for tr in sc.obstacle_tr:
            nrm, o0 = tr[[2, 5, 8]], tr[9:]
            side = np.where((x - o0) @ nrm >= 0, 1.0, -1.0)[:, None] * nrm
            pa = x - r * side
            gap = ((pa - o0) * side).sum(1)
            k = np.flatnonzero(gap < 0)
            pb = pa[k] - gap[k, None] * side[k]
            cp = 0.5 * (pa[k] + pb)
            lever = cp if case["quirks"] else cp - x[k]
            f, t = _hooke(row, pb - pa[k], v[k] + np.cross(w[k], lever), 0.5 * m, 2 * math.sqrt(row[0] / (0.5 * m)),
                          cp - x[k])
            F[k] += f
            M[k] += t
        F += m * np.array([0, 0, -9.81])
        x = x + dt * v
        v = v + dt * F / m
        s = np.linalg.norm(w, axis=1, keepdims=True)
        dq = np.concatenate([np.sin(0.5 * dt * s) / np.maximum(s, 1e-300) * w, np.cos(0.5 * dt * s)], 1)
        q = _qmul(dq, q)
        w = w + dt * M / inertia
    out = {"pos": x, "quat": q, "vel": v, "omega": w, "contacts": None}
    if case["form"] == "driver":
        out.update(force=F, torque=M)
    return out
