"""Performance cases of the coupled LB/DEM step, through the public binding (lbm-dem_amd/python).

A case is one piece of work that a program using the library repeats: the steps of one output
interval and the reads that follow it, a set of runs served by the run pool, or a fluid-only flow.
Kinds:

  run    one impact run: ``lbdem_cycle`` over an output interval, then the records that a program
         writes (impactors, walls, fluid mass, particles; with ``fields`` also the node fields)
  steps  the same run driven as the reference's main loop drives it: one call per sub-step
         (DEM, coupling, LB, free surface) with the stress diagnostics on, then the screen output
  pool   requests submitted to a run pool, each on a stream of its own, and waited for: set-up, steps
         and results of every run
  fluid  no spheres, impactor or free surface: forced flow in a periodic or closed box

``prec`` is the storage precision of the populations (fp64, fp32, fp16). Runs with single- or
half-precision populations hand their results on in single precision, as a program does that writes
what such a run computes.
"""
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lbm-dem_amd", "python"))
import lbdem  # noqa: E402
import workloads  # noqa: E402

PREC = {"fp64": lbdem.PREC_FP64, "fp32": lbdem.PREC_FP32, "fp16": lbdem.PREC_FP16}
ELT = {"fp64": 8, "fp32": 4, "fp16": 2}
WARM = 24  # start-up steps of every context: the tile tuner's launches and the first list rebuilds


def listed():
    return [
        # a drop test watched step by step: the smallest box the tests use, one step and a record per
        # call; latency of launches and reads
        dict(name="drop14_fp32", kind="run", prec="fp32", X=14, Y=20, Z=14, fill=11.0, n=0, r=2.0, rImp=3.0,
             speed=0.02, periodic=False, steps=1, particles=False, fields=False, model="NEWTONIAN", turb=0.0),
        # the reference's main loop on the reference-scale box (64^3, 480 spheres of radius 3,
        # impactor of radius 8) in double precision, a screen output every 20 steps
        dict(name="loop64_fp64", kind="steps", prec="fp64", X=64, Y=64, Z=64, fill=48.0, n=480, r=3.0, rImp=8.0,
             speed=0.005, periodic=True, steps=20, particles=True),
        # the same box through lbdem_cycle in single precision, the interactive or sweep size
        dict(name="impact64_fp32", kind="run", prec="fp32", X=64, Y=64, Z=64, fill=48.0, n=480, r=3.0, rImp=8.0,
             speed=0.005, periodic=True, steps=50, particles=True, fields=False, model="NEWTONIAN", turb=0.0),
        # an odd-sized closed box in double precision whose mass, density and type fields are
        # written out every 40 steps (the fluid files)
        dict(name="closed91_fp64", kind="run", prec="fp64", X=91, Y=117, Z=83, fill=88.0, n=900, r=3.5, rImp=9.0,
             speed=0.01, periodic=False, steps=40, particles=True, fields=True, model="NEWTONIAN", turb=0.0),
        # the largest box of the batched workload on its own
        dict(name="impact128_fp32", kind="run", prec="fp32", X=128, Y=128, Z=128, fill=96.0, n=2300, r=3.5, rImp=25.6,
             speed=0.01, periodic=True, steps=100, particles=True, fields=False, model="NEWTONIAN", turb=0.0),
        # a yield-stress fluid with the turbulence term, uneven box sides (per-node viscosity)
        dict(name="bingham150_fp32", kind="run", prec="fp32", X=150, Y=110, Z=100, fill=80.0, n=1500, r=4.0, rImp=10.0,
             speed=0.01, periodic=True, steps=50, particles=True, fields=False, model="BINGHAM", turb=0.05),
        # the headline impact run (256 x 320 x 256, 31 000 spheres of radius 4, impactor of radius
        # 16) in the three storage precisions, records every 100 (50) steps
        dict(name="impact256_fp32", kind="run", prec="fp32", X=256, Y=320, Z=256, fill=256.0, n=31000, r=4.0, rImp=16.0,
             speed=0.01, periodic=True, steps=100, particles=True, fields=False, model="NEWTONIAN", turb=0.0),
        dict(name="impact256_fp64", kind="run", prec="fp64", X=256, Y=320, Z=256, fill=256.0, n=31000, r=4.0, rImp=16.0,
             speed=0.01, periodic=True, steps=50, particles=True, fields=False, model="NEWTONIAN", turb=0.0),
        dict(name="impact256_fp16", kind="run", prec="fp16", X=256, Y=320, Z=256, fill=256.0, n=31000, r=4.0, rImp=16.0,
             speed=0.01, periodic=True, steps=100, particles=True, fields=False, model="NEWTONIAN", turb=0.0),
        # a service or parameter sweep: 10 requests of edge 64-128 and 100-400 steps that arrive together
        dict(name="pool10_fp32", kind="pool", prec="fp32", boxes=10, lo=64, hi=128, stepsLo=100, stepsHi=400),
        # channel flow without spheres, free surface or impactor
        dict(name="channel160_fp32", kind="fluid", prec="fp32", X=160, Y=130, Z=98, periodic=True, steps=300, turb=0.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_steps(rng, nodes, lo, hi):
    """Steps of one pass, fewer in larger boxes: at most the node updates of 50 steps of the largest box."""
    return max(1, min(_log_int(rng, lo, hi), int(5.0e8 / nodes)))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "run", "steps", "steps", "fluid", "fluid", "pool"])
    if kind == "pool":
        lo = rng.randint(48, 70)
        return dict(kind="pool", prec=rng.choice(["fp32", "fp32", "fp16"]), boxes=rng.randint(2, 10), lo=lo,
                    hi=rng.randint(72, 120), stepsLo=rng.randint(20, 100), stepsHi=rng.randint(120, 300))
    if kind == "fluid":
        X, Y, Z = (_log_int(rng, 9, 170) for _ in range(3))
        return dict(kind="fluid", prec=rng.choice(["fp32", "fp32", "fp64"]), X=X, Y=Y, Z=Z,
                    periodic=rng.random() < 0.6, steps=_log_steps(rng, X * Y * Z, 10, 200),
                    turb=rng.choice([0.0, 0.0, 0.05, 0.5]))
    X, Z = _log_int(rng, 14, 250), _log_int(rng, 14, 250)
    Y = _log_int(rng, 20, 300)
    fill = round(rng.uniform(0.6, 0.8) * Y, 1)
    r = round(rng.uniform(2.0, 4.0), 2)
    rImp = round(max(2.2, rng.uniform(0.06, 0.2) * min(X, Y, Z)), 2)
    phi = rng.uniform(0.1, 0.48)
    bed = min(fill, _impactor_y(Y, fill, rImp) - rImp - 1.0) - 1.0
    n = 0
    if min(X - 2, Z - 2, bed) > 2.5 * r:
        n = int(phi * (X - 2) * (Z - 2) * bed / (4.0 / 3.0 * math.pi * r ** 3))
    case = dict(kind=kind, prec=rng.choice(["fp64", "fp32", "fp32", "fp16"]), X=X, Y=Y, Z=Z, fill=fill, n=n, r=r,
                rImp=rImp, speed=round(rng.uniform(0.002, 0.02), 4), periodic=rng.random() < 0.6,
                steps=_log_steps(rng, X * Y * Z, 1 if kind == "run" else 4, 100), particles=rng.random() < 0.7)
    if kind == "run":
        case.update(fields=X * Y * Z < 600000 and rng.random() < 0.5,
                    model=rng.choice(["NEWTONIAN", "NEWTONIAN", "NEWTONIAN", "BINGHAM"]), turb=rng.choice([0.0, 0.0, 0.05]))
    return case


# ----------------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------------
def _impactor_y(Y, fill, r):
    """The impactor starts half a radius deep, or as high as the lid lets it."""
    return min(Y - r - 3.0, fill + 0.5 * r)


def _impact(case, seed):
    """Values, spheres and impactor of an impact run: a seeded packing below a partly immersed impactor."""
    X, Y, Z = case["X"], case["Y"], case["Z"]
    y = _impactor_y(Y, case["fill"], case["rImp"])
    n = case["n"]
    while True:
        try:
            v, ps, obs = workloads.impact_box(
                size=(X, Y, Z), fluid_height=case["fill"], n_spheres=n, r=case["r"], r_imp=case["rImp"], y_imp=y,
                speed=case["speed"], seed=seed, relax=60, periodic=case["periodic"],
                bed_top=min(case["fill"], y - case["rImp"] - 1.0))
            break
        except RuntimeError:  # a narrow bed holds fewer spheres
            n = int(0.9 * n)
    rng = np.random.default_rng(seed)
    obs.x0 = obs.x0 + rng.uniform(-0.5, 0.5, size=(1, 3))
    v["maxTime"] = 1.0e9
    if case.get("model") == "BINGHAM":
        v.update(rheologyModel="BINGHAM", plasticVisc=0.08, yieldStress=2.0e-5)
    if case.get("turb"):
        v.update(turbulenceSolve=1, turbConst=case["turb"])
    return v, ps, obs


def _fluid(case, seed):
    """Values of a forced flow: body force, initial velocity and viscosity from the seed."""
    rng = np.random.default_rng(seed)
    v = dict(lbdem.DEFAULTS)
    F, u = rng.uniform(-2.0e-5, 2.0e-5, 3), rng.uniform(-0.03, 0.03, 3)
    v.update(lbSolve=1, demSolve=0, freeSurfaceSolve=0, forceFieldSolve=1, maxTime=1.0e9,
             lbSizeX=float(case["X"]), lbSizeY=float(case["Y"]), lbSizeZ=float(case["Z"]), rheologyModel="NEWTONIAN",
             initVisc=float(rng.uniform(0.02, 0.2)), lbFX=float(F[0]), lbFY=float(F[1]), lbFZ=float(F[2]),
             initVelocityX=float(u[0]), initVelocityY=float(u[1]), initVelocityZ=float(u[2]), density=2.5,
             objectDensity=3.0)
    side = 4 if case["periodic"] else 7
    v.update(boundary0=side, boundary1=side, boundary2=7, boundary3=7, boundary4=side, boundary5=side)
    if case["turb"]:
        v.update(turbulenceSolve=1, turbConst=case["turb"])
    return v


def _sim(v, ps, obs, prec, stress=False):
    sim = lbdem.Simulation(lbdem.Library.load(), lbdem.params_from_values(v, PREC[prec]), ps, obs)
    if stress:
        sim.set_stress()
    sim.init()
    return sim


def _many(case, seed):
    """Boxes of the served workload: edges spread over [lo, hi], the rest drawn from the seed."""
    rng = np.random.default_rng(seed)
    n = case["boxes"]
    edges = [int(round(case["lo"] + (case["hi"] - case["lo"]) * k / max(n - 1, 1))) for k in range(n)]
    return [workloads.random_impact_run(rng, (e,), 1, relax=40) for e in edges], rng


def _step(sim):
    sim.dem_step()
    sim.coupling_step()
    sim.lb_step()
    sim.fs_step()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pool":
        runs, rng = _many(case, seed)
        reqs = [(lbdem.params_from_values(r.values, PREC[case["prec"]]), r.particles, r.objects,
                 int(rng.integers(case["stepsLo"], case["stepsHi"] + 1))) for r in runs]
        pool = lbdem.Pool(lbdem.Library.load(), budget_bytes=8 << 30, max_concurrent=16, steps_per_chunk=32,
                          batching=False)
        return dict(case=case, pool=pool, reqs=reqs)
    if kind == "fluid":
        sim = _sim(_fluid(case, seed), lbdem.ParticleSet(), lbdem.ObjectSet(), case["prec"])
        sim.cycle(WARM)
    elif kind == "steps":
        sim = _sim(*_impact(case, seed), case["prec"], stress=True)
        for _ in range(WARM):
            _step(sim)
    else:
        sim = _sim(*_impact(case, seed), case["prec"])
        sim.cycle(WARM)
    sim.synchronize()
    return dict(case=case, sim=sim)


# ----------------------------------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------------------------------
def _hand_on(case, out):
    if case["prec"] == "fp64":
        return out
    return {k: np.asarray(a, np.float32) for k, a in out.items()}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "pool":
        ids = [state["pool"].submit(*q) for q in state["reqs"]]
        res = [state["pool"].wait(i) for i in ids]
        if any(r["state"] != lbdem.RUN_DONE for r in res):
            raise RuntimeError("a run of the pool failed: %s" % [r["message"] for r in res if r["message"]])
        return _hand_on(case, dict(objects=np.concatenate([r["objects"] for r in res]),
                                   mass=np.array([r["totalMass"] for r in res])))
    sim = state["sim"]
    if kind == "fluid":
        sim.cycle(case["steps"] - 1)
        sim.store_velocity()
        sim.cycle(1)
        u, visc = sim.velocity()
        out = dict(u=u, walls=sim.walls())
        if case["turb"]:
            out["visc"] = visc
        return _hand_on(case, out)
    if kind == "steps":
        for _ in range(case["steps"]):
            _step(sim)
    else:
        sim.cycle(case["steps"])
    out = dict(objects=sim.objects(), walls=sim.walls(), mass=np.array([sim.total_mass()]))
    if case["particles"]:
        out["particles"] = sim.particles()
    if kind == "steps":
        out["stress"] = sim.stress()[0]
    elif case["fields"]:
        _, out["nodeMass"], out["nodeDensity"] = sim.fields(want_f=False)
    return _hand_on(case, out)


# ----------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------
def _box_work(active, spheres, steps, prec):
    """Populations of every active node read and written and its type read, once a step; per sphere
    its state (positions, velocities, hydrodynamic sums, contact history of about six contacts)."""
    elt = ELT[prec]
    return np.array([steps * (active * (38.0 * elt + 1.0) + spheres * 700.0),
                     steps * (active * 250.0 + spheres * 12.0 * 300.0)])


def work(case):
    kind, prec = case["kind"], case["prec"]
    if kind == "pool":
        n, steps = case["boxes"], 0.5 * (case["stepsLo"] + case["stepsHi"])
        w = np.zeros(2)
        for k in range(n):
            e = case["lo"] + (case["hi"] - case["lo"]) * k / max(n - 1, 1)
            w += _box_work(0.7 * (e - 2.0) ** 2 * e, 0.25 * e * (e - 2.0) ** 2 * 0.42 / 180.0, steps, prec)
    elif kind == "fluid":
        w = _box_work((case["X"] - 2.0) * (case["Y"] - 2.0) * (case["Z"] - 2.0), 0, case["steps"], prec)
    else:
        w = _box_work((case["X"] - 2.0) * case["fill"] * (case["Z"] - 2.0), case["n"], case["steps"], prec)
    return {"bytes": float(w[0]), "flops": float(w[1])}


# ----------------------------------------------------------------------------------------------
# the same in 64 bits: the fluid cases (the coupled cases have no plain formula: their results come
# from free-surface, sphere and contact events over many steps)
# ----------------------------------------------------------------------------------------------
_C = np.array([(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
               (-1, 1, 0), (1, -1, 0), (0, 1, 1), (0, -1, -1), (0, -1, 1), (0, 1, -1), (1, 0, 1), (-1, 0, -1),
               (1, 0, -1), (-1, 0, 1)])
_W = np.array([1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12)
_OPP = [0] + [q + 1 if q % 2 else q - 1 for q in range(1, 19)]


def exact(case, seed):
    """D3Q19 BGK with Guo forcing and half-way bounce-back in 64-bit torch: velocity of every node and
    the momentum each wall took in the last step (and the node viscosity with the Smagorinsky term)."""
    if case["kind"] != "fluid":
        return None
    import torch
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    v = _fluid(case, seed)
    X, Y, Z = case["X"], case["Y"], case["Z"]
    F = [v["lbFX"], v["lbFY"], v["lbFZ"]]
    u0 = [v["initVelocityX"] + 0.5 * F[0], v["initVelocityY"] + 0.5 * F[1], v["initVelocityZ"] + 0.5 * F[2]]
    shape = (Z - 2, Y - 2, X - 2)  # the nodes inside the boundary layer
    wall = [v["boundary%d" % i] == 7 for i in range(6)]
    axis = {0: 2, 1: 1, 2: 0}  # x, y, z as tensor axes

    def cdot(q, a):
        return sum(float(_C[q][k]) * a[k] for k in range(3) if _C[q][k])

    def feq(q, n, u, usq):
        cu = cdot(q, u)
        return _W[q] * n * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * usq)

    one = torch.ones(shape, dtype=torch.float64, device=dev)
    uu = [one * c for c in u0]
    f = torch.stack([feq(q, one, uu, sum(c * c for c in uu)) * one for q in range(19)])
    # which wall a link that leaves through the boundary layer meets (the last one that holds the node)
    number = np.full((Z, Y, X), -1)
    k = 0
    for i in range(6):
        if wall[i]:
            sl = [slice(None)] * 3
            sl[axis[i // 2]] = 0 if i % 2 == 0 else -1
            number[tuple(sl)] = k
            k += 1
    links = []
    for q in range(1, 19):
        c = _C[q]
        idx = [np.arange(1, m - 1) + c[a] for m, a in ((Z, 2), (Y, 1), (X, 0))]
        for m, a, j in ((Z, 2, 0), (Y, 1, 1), (X, 0, 2)):  # periodic axes wrap inside the layer
            if not wall[2 * a]:
                idx[j] = (idx[j] - 1) % (m - 2) + 1
        links.append(torch.from_numpy(number[np.ix_(*idx)]).to(dev))
    turb = case["turb"]
    nu = one * v["initVisc"]
    steps = WARM + case["steps"]
    walls = np.zeros((k, lbdem.W["REC"]))
    for s in range(steps):
        n = f.sum(0)
        j = [sum(float(_C[q][a]) * f[q] for q in range(19) if _C[q][a]) for a in range(3)]
        u = [(j[a] + 0.5 * F[a]) / n for a in range(3)]
        usq = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
        eq = [feq(q, n, u, usq) for q in range(19)]
        if turb:
            t = {}
            for a in range(3):
                for b in range(a, 3):
                    t[a, b] = sum(float(_C[q][a] * _C[q][b]) * (f[q] - eq[q]) for q in range(19) if _C[q][a] * _C[q][b])
                    t[a, b] = t[a, b] * 1.5 / ((0.5 + 3.0 * nu) * n)
            mag = 0.5 * (t[0, 0] ** 2 + t[1, 1] ** 2 + t[2, 2] ** 2 + 2.0 * (t[0, 1] ** 2 + t[0, 2] ** 2 + t[1, 2] ** 2))
            nu = torch.clamp(v["initVisc"] + turb * 2.0 * torch.sqrt(mag), (0.500001 - 0.5) / 3.0, (1.8 - 0.5) / 3.0)
        om, omf = 1.0 / (0.5 + 3.0 * nu), 1.0 - 1.0 / (1.0 + 6.0 * nu)
        uF = sum(u[a] * F[a] for a in range(3))
        new = torch.empty_like(f)
        last = s == steps - 1
        for q in range(19):
            cu, cF = cdot(q, u), cdot(q, F)
            post = f[q] + om * (eq[q] - f[q]) + omf * _W[q] * (9.0 * cu * cF + 3.0 * (cF - uF))
            if q == 0:
                new[0] = post
                continue
            meets = links[q - 1]
            bounce = meets >= 0
            dims = [axis[a] for a in range(3) if _C[q][a]]
            moved = torch.roll(post, [int(_C[q][a]) for a in range(3) if _C[q][a]], dims)
            # a slot whose upstream neighbour is a wall node keeps what that link reflects
            back = links[_OPP[q] - 1] >= 0
            new[q] = torch.where(back, new[q], moved) if q > _OPP[q] else torch.where(back, torch.zeros_like(moved), moved)
            if q < _OPP[q]:
                first = post
            else:
                p = _OPP[q]  # the pair (p, q): each reflects into the other
                new[q] = torch.where(back, first, new[q])
                new[p] = torch.where(bounce, post, new[p])
            if last and k:
                got = torch.zeros(k + 1, dtype=torch.float64, device=dev)
                got.index_add_(0, (meets + 1).reshape(-1), (2.0 * (post - _W[q])).reshape(-1))
                walls[:, lbdem.W["FHYDRO"]:lbdem.W["FHYDRO"] + 3] += got[1:].cpu().numpy()[:, None] * _C[q]
        f = new
    full = torch.zeros((Z, Y, X, 3), dtype=torch.float64, device=dev)
    full[1:-1, 1:-1, 1:-1] = torch.stack(u, dim=-1)
    out = dict(u=full.reshape(-1, 3), walls=walls if k else None)
    if turb:
        visc = torch.zeros((Z, Y, X), dtype=torch.float64, device=dev)
        visc[1:-1, 1:-1, 1:-1] = nu
        out["visc"] = visc.reshape(-1)
    return out
