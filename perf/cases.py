"""What a user of this framework has it do, as measurable cases: predictor-corrector runs of fluid, gas and
solid bodies in both precisions, single derivative evaluations, ensembles, N-body runs, the direct sum, SPH
with self-gravity, and the gradient of a gas run.

A case is a dict of plain values.  `prepare` builds the resident solver a program keeps, `run` is one pass
through the public entry points (the Python classes, and the C ABI's getters into host buffers that the
program keeps), `work` is what a pass cannot do without, and `exact` restates the gas and gravity paths in
64-bit torch.  Every kind steps a resident state, so a pass goes on from where the last one ended; the
inputs are chosen so that hundreds of passes leave the bodies in the same regime.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from opensph_amd import gpu, initial
from opensph_amd.gravity import GpuGravity
from opensph_amd.state import ParticleState, RunConfig, basalt

G = 6.67408e-11  # Constants::gravity

# Flops of one unordered pair of the solid term set; of a particle pair and of a quadrupole and an octupole
# expansion of the tree walk, with their counts per particle at theta 0.5 and leaves of up to 25 particles.
FLOP_SPH_PAIR = 198.0
SPH_PAIRS_PER_PARTICLE = 33.0
FLOP_GRAVITY_PAIR = 22.0
FLOP_EXPANSION = {"quadrupole": 61.0, "octupole": 140.0}
TREE_PAIRS, TREE_EXPANSIONS = 1600.0, 650.0
STATE_BYTES = 612.0  # per particle and step: the state's planes read and written once


def listed():
    return [
        # the smallest run in use: a fluid sphere of two thousand particles, bound by launches and host waits
        dict(name="fluid_2k_fp64", kind="gas", n=2000, bodies=1, precision="fp64", steps=10, gravity=False),
        # two gas bodies of ordinary size in mixed precision
        dict(name="gas_40k_mixed", kind="gas", n=40000, bodies=2, precision="mixed", steps=10, gravity=False),
        # the headline: a million-particle solid impact with damage, in contact, in both precisions
        dict(name="impact_1M_mixed", kind="impact", n=1000000, precision="mixed", steps=40),
        dict(name="impact_1M_fp64", kind="impact", n=1000000, precision="fp64", steps=25),
        # one derivative evaluation, as a host integrator that steps the state itself asks for it
        dict(name="evaluate_531k_fp64", kind="evaluate", n=531277, precision="fp64"),
        # a parameter study: impacts of 5k to 200k particles stepped together
        dict(name="ensemble_16_mixed", kind="ensemble", members=16, n_lo=5000, n_hi=200000, precision="mixed", steps=10),
        # Barnes-Hut N-body runs: large in mixed precision, ordinary in FP64, small with octupoles
        dict(name="nbody_8M_mixed", kind="nbody", n=8000000, order="quadrupole", theta=0.5, leaf=25,
             precision="mixed", steps=4),
        dict(name="nbody_1M_fp64", kind="nbody", n=1000003, order="quadrupole", theta=0.5, leaf=25,
             precision="fp64", steps=5),
        dict(name="nbody_20k_fp64", kind="nbody", n=20011, order="octupole", theta=0.5, leaf=25,
             precision="fp64", steps=5),
        # the exact self-gravity of a small system
        dict(name="direct_12k_fp64", kind="direct", n=12345),
        # self-gravitating bodies: SPH with Barnes-Hut gravity in every evaluation
        dict(name="gas_gravity_100k_mixed", kind="gas", n=100000, bodies=2, precision="mixed", steps=5, gravity=True),
        # the gradient of a gas run: forward with checkpoints, then backward
        dict(name="adjoint_10k_fp64", kind="adjoint", n=10619, precision="fp64", steps=20, checkpoint=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gas", "gas", "impact", "evaluate", "ensemble", "nbody", "nbody", "direct", "adjoint"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "gas":
        gravity = rng.random() < 0.4
        return dict(kind="gas", n=_log_int(rng, 1500, 150000), bodies=rng.choice([1, 2]), precision=precision,
                    steps=rng.choice([5, 8, 10]), gravity=gravity)
    if kind == "impact":
        return dict(kind="impact", n=_log_int(rng, 5000, 1000000), precision=precision, steps=rng.choice([10, 15, 20]))
    if kind == "evaluate":
        return dict(kind="evaluate", n=_log_int(rng, 2000, 900000), precision=precision)
    if kind == "ensemble":
        return dict(kind="ensemble", members=rng.randrange(3, 17), n_lo=5000, n_hi=_log_int(rng, 20000, 200000),
                    precision=precision, steps=rng.choice([5, 8, 10]))
    if kind == "nbody":
        return dict(kind="nbody", n=_log_int(rng, 1000, 4000000), order=rng.choice(["quadrupole", "octupole"]),
                    theta=round(rng.uniform(0.45, 0.9), 3), leaf=rng.choice([10, 25, 25, 40]), precision=precision,
                    steps=rng.choice([2, 3, 4]))
    if kind == "direct":
        return dict(kind="direct", n=_log_int(rng, 500, 30000))
    return dict(kind="adjoint", n=_log_int(rng, 3000, 100000), precision=precision, steps=rng.choice([8, 12, 20]),
                checkpoint=rng.choice([4, 10]))


# ---- inputs -------------------------------------------------------------------------------------------------


def _lattice_sphere(n, radius):
    """About n points of a hexagonal close packing inside a sphere about the origin, and their spacing h."""
    h = (4.0 / 3.0 * math.pi * radius ** 3 / n) ** (1.0 / 3.0)
    dx = 1.1 * h
    k = int(radius / dx) + 3
    i = np.arange(-k, k + 1)
    I, J, K = np.meshgrid(i, i, np.arange(-2 * k, 2 * k + 1), indexing="ij")
    x = (I + 0.5 * ((J + K) % 2)) * dx
    y = (J * math.sqrt(3.0) / 2.0 + (K % 2) * math.sqrt(3.0) / 6.0) * dx
    z = K * math.sqrt(6.0) / 3.0 * dx
    p = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    return p[np.einsum("ij,ij->i", p, p) <= radius * radius], h


def _gas_inputs(case, seed):
    """One or two basalt bodies as gas (no stress): positions with h in lane 3, velocities with noise, mass,
    density, energy, body flag, and the first time step.  Two bodies touch and approach each other; bodies
    with gravity are of planetesimal size."""
    rng = np.random.default_rng(seed)
    gravity = bool(case.get("gravity"))
    radius = 4.0e5 if gravity else 1000.0
    speed = 2000.0 if gravity else 100.0
    two = case.get("bodies", 2) == 2
    n_first = case["n"] / 1.125 if two else case["n"]
    p, h = _lattice_sphere(n_first, radius)
    v = np.zeros((len(p), 3))
    flag = np.zeros(len(p), dtype=np.uint32)
    if two:  # half the radius at the same spacing
        q, _ = _lattice_sphere(case["n"] - n_first, 0.5 * radius)
        q[:, 0] += radius + 0.5 * radius + 0.5 * h
        w = np.zeros((len(q), 3))
        w[:, 0] = -speed
        p, v = np.concatenate([p, q]), np.concatenate([v, w])
        flag = np.concatenate([flag, np.ones(len(q), dtype=np.uint32)])
    n = len(p)
    p = p + rng.normal(0.0, 0.01 * h, size=(n, 3))
    v = v + rng.normal(0.0, 1.0, size=(n, 3))
    eta = 1.3 * h
    rho0 = 2700.0
    m = np.full(n, rho0 * (1.1 * h) ** 3 / math.sqrt(2.0))  # the lattice's volume per point
    return dict(r=np.concatenate([p, np.full((n, 1), eta)], axis=1), v=np.concatenate([v, np.zeros((n, 1))], axis=1),
                m=m, rho=np.full(n, rho0), u=rng.uniform(0.9e3, 1.1e3, n), flag=flag, dt=0.1 * eta / 3200.0)


def _gas_state(a):
    st = ParticleState(len(a["m"]), [basalt()])
    for k in ("r", "v", "m", "rho", "u", "flag"):
        st[k] = a[k]
    st["reduce"] = 1.0
    return st


def _gas_config(case, a):
    return RunConfig(solid_stress=0, adaptive_h=0, has_reduce=0, has_damage=0, criteria=1, initial_dt=a["dt"],
                     gravity=2 if case.get("gravity") else 0)


def _impact(precision, seed, **kw):
    """A solid impact built on the device, the bodies in contact, with the seed's flaws and velocity noise."""
    s = initial.device_impact(precision=precision, flaw_seed=seed, offset_h=0.5, **kw)
    v = np.empty((s.n, 4))
    _get(s, "POSITION", 1, v)
    v[:, :3] += np.random.default_rng(seed).normal(0.0, 1.0, size=(s.n, 3))
    s._check(s.L.osph_set_quantity(s.ctx, gpu.Q["POSITION"], 1, v.ctypes.data, 0), "osph_set_quantity")
    s.dt = 1.0e-3
    return s


def _nbody_inputs(case, seed):
    """A uniform sphere of equal masses with random virial velocities."""
    rng = np.random.default_rng(seed)
    n, radius, total = case["n"], 1.0e5, 1.0e19
    d = rng.standard_normal((n, 3))
    d *= (radius * rng.random(n) ** (1.0 / 3.0) / np.sqrt(np.einsum("ij,ij->i", d, d)))[:, None]
    speed = math.sqrt(G * total / radius / 3.0)
    v = np.zeros((n, 4))
    v[:, :3] = rng.standard_normal((n, 3)) * (0.6 * speed)
    r = np.empty((n, 4))
    r[:, :3] = d
    r[:, 3] = 10.0
    return r, v, np.full(n, total / n)


NBODY_DT = 0.5


# ---- preparation and passes -----------------------------------------------------------------------------------


def _get(s, quantity, order, out):
    s._check(s.L.osph_get_quantity(s.ctx, gpu.Q[quantity], order, out.ctypes.data, 0), "osph_get_quantity")
    return out


def _snapshot_buffers(n):
    return dict(r=np.zeros((n, 4)), v=np.zeros((n, 4)), rho=np.zeros(n), u=np.zeros(n))


def _snapshot(s, out):
    _get(s, "POSITION", 0, out["r"])
    _get(s, "POSITION", 1, out["v"])
    _get(s, "DENSITY", 0, out["rho"])
    _get(s, "ENERGY", 0, out["u"])
    return out


def _sized_impact(n):
    return dict(n_target=int(0.95 * n), n_projectile=max(60, int(0.05 * n)))


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case)
    if kind == "gas":
        a = _gas_inputs(case, seed)
        s = gpu.GpuSolver(_gas_state(a), _gas_config(case, a), precision=case["precision"])
        state.update(solver=s, out=_snapshot_buffers(s.n))
    elif kind == "impact":
        s = _impact(case["precision"], seed, **_sized_impact(case["n"]))
        state.update(solver=s, out=_snapshot_buffers(s.n))
    elif kind == "evaluate":
        a = _gas_inputs(dict(case, bodies=2), seed)
        s = gpu.GpuSolver(_gas_state(a), _gas_config(case, a), precision=case["precision"])
        n = s.n
        state.update(solver=s, out=dict(dv=np.zeros((n, 4)), drho=np.zeros(n), du=np.zeros(n),
                                        ncnt=np.zeros(n, dtype=np.uint32)))
    elif kind == "ensemble":
        rng = np.random.default_rng([seed, 7])
        # the sizes are the study's own; the seed draws angles, speeds, flaws and noise
        sizes = np.exp(np.linspace(math.log(case["n_lo"]), math.log(case["n_hi"]), case["members"]))
        ms = []
        for k, n in enumerate(sizes):
            ratio = 0.1
            n_p = max(100, int(n * ratio ** 3 / (1 + ratio ** 3)))
            ms.append(_impact(case["precision"], seed + 31 * k, n_target=int(n) - n_p, n_projectile=n_p,
                              r_projectile=50e3 * ratio, speed=rng.uniform(3e3, 7e3), angle_deg=rng.uniform(10.0, 80.0)))
        state.update(solvers=ms, out=[dict(r=np.zeros((s.n, 4)), v=np.zeros((s.n, 4))) for s in ms])
    elif kind == "nbody":
        r, v, m = _nbody_inputs(case, seed)
        g = GpuGravity(r, m, v, theta=case["theta"], order=case["order"], leaf_size=case["leaf"], G=G,
                       precision=case["precision"])
        state.update(gravity=g, out=dict(r=np.zeros((g.n, 4)), v=np.zeros((g.n, 4))))
    elif kind == "direct":
        r, v, m = _nbody_inputs(case, seed)
        r[:, 3] = 2.0e3  # softening supports that overlap their neighbours
        state.update(gravity=GpuGravity(r, m, solver="brute_force", G=G))
    elif kind == "adjoint":
        a = _gas_inputs(dict(case, bodies=2), seed)
        s = gpu.GpuSolver(_gas_state(a), _gas_config(case, a), precision=case["precision"])
        seed_r, seed_v, seed_u = _objective(a)
        state.update(solver=s, dts=np.full(case["steps"], a["dt"]), seed_r=seed_r, seed_v=seed_v, seed_u=seed_u)
    else:
        raise ValueError(kind)
    return state


def _objective(a):
    """dJ/d(final r, v, u) of J = (the impactor's momentum along its path and across it, its centre's
    distance, and the heat of both bodies), scaled to comparable sizes."""
    n = len(a["m"])
    w = (a["flag"] == 1) / max(1, int(np.sum(a["flag"] == 1)))
    seed_r, seed_v = np.zeros((n, 3)), np.zeros((n, 3))
    seed_r[:, 0], seed_r[:, 1] = 0.1 * w, 0.05 * w
    seed_v[:, 0], seed_v[:, 1] = w, 0.3 * w
    return seed_r, seed_v, np.full(n, 1.0e-3 / n)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("gas", "impact"):
        s = state["solver"]
        for _ in range(case["steps"]):
            s.step()
        return _snapshot(s, state["out"])
    if kind == "evaluate":
        s, out = state["solver"], state["out"]
        s.integrate()
        _get(s, "POSITION", 2, out["dv"])
        _get(s, "DENSITY", 1, out["drho"])
        _get(s, "ENERGY", 1, out["du"])
        _get(s, "NEIGHBOR_CNT", 0, out["ncnt"])
        return out
    if kind == "ensemble":
        for _ in range(case["steps"]):
            gpu.step_batch(state["solvers"])
        for s, out in zip(state["solvers"], state["out"]):
            _get(s, "POSITION", 0, out["r"])
            _get(s, "POSITION", 1, out["v"])
        return state["out"]
    if kind == "nbody":
        g, out = state["gravity"], state["out"]
        g.leapfrog(NBODY_DT, case["steps"])
        g._check(g.L.osph_gravity_get(g.ctx, 0, out["r"].ctypes.data, 32), "osph_gravity_get")
        g._check(g.L.osph_gravity_get(g.ctx, 1, out["v"].ctypes.data, 32), "osph_gravity_get")
        return out
    if kind == "direct":
        g = state["gravity"]
        g.build()
        dv, _ = g.eval_self()
        return dict(dv=dv)
    s = state["solver"]
    s.adjoint_forward(state["dts"], case["checkpoint"])
    grads = s.adjoint_backward(seed_r=state["seed_r"], seed_v=state["seed_v"], seed_u=state["seed_u"])
    return {k: grads[k] for k in ("r", "v", "rho", "u", "eos")}


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    tree = FLOP_GRAVITY_PAIR * TREE_PAIRS + FLOP_EXPANSION["octupole"] * TREE_EXPANSIONS
    if kind in ("gas", "impact"):
        flops = n * FLOP_SPH_PAIR * SPH_PAIRS_PER_PARTICLE + (n * tree if case.get("gravity") else 0.0)
        return dict(bytes=case["steps"] * n * STATE_BYTES + 80.0 * n, flops=case["steps"] * flops)
    if kind == "evaluate":
        return dict(bytes=n * 200.0, flops=n * FLOP_SPH_PAIR * SPH_PAIRS_PER_PARTICLE)
    if kind == "ensemble":
        total = float(np.sum(np.exp(np.linspace(math.log(case["n_lo"]), math.log(case["n_hi"]), case["members"]))))
        return dict(bytes=case["steps"] * total * STATE_BYTES + 64.0 * total,
                    flops=case["steps"] * total * FLOP_SPH_PAIR * SPH_PAIRS_PER_PARTICLE)
    if kind == "nbody":
        tree = FLOP_GRAVITY_PAIR * TREE_PAIRS + FLOP_EXPANSION[case["order"]] * TREE_EXPANSIONS
        tree *= min(1.0, (0.5 / case["theta"]) ** 2) * min(1.0, n / 20000.0)
        return dict(bytes=case["steps"] * n * 200.0 + 64.0 * n, flops=case["steps"] * n * tree)
    if kind == "direct":
        return dict(bytes=n * 64.0, flops=FLOP_GRAVITY_PAIR * n * n)
    # forward, replay and reverse: three evaluations a step, the reverse one of twice the flops
    return dict(bytes=case["steps"] * n * 3 * STATE_BYTES, flops=case["steps"] * n * 4 * FLOP_SPH_PAIR * SPH_PAIRS_PER_PARTICLE)


# ---- the same in 64 bits, in torch --------------------------------------------------------------------------


def _m4_table():
    """The tabulated gradient factor of the M4 spline: 40001 values uniform in q^2 over [0, 4]."""
    q = np.sqrt(np.arange(40001) / 10000.0)
    with np.errstate(divide="ignore", invalid="ignore"):
        inner = -0.75 * (2.0 - q) ** 2 + 3.0 * (1.0 - q) ** 2
        g = np.where(q < 1.0, inner, -0.75 * (2.0 - q) ** 2) / (np.pi * q)
    g[0] = -3.0 / np.pi
    g[-1] = 0.0
    return g


def _softening_table():
    """The tabulated gradient factor of the gravity kernel of the M4 spline."""
    q = np.sqrt(np.arange(40001) / 10000.0)
    with np.errstate(divide="ignore", invalid="ignore"):
        inner = 4.0 / 3.0 * q - 6.0 / 5.0 * q ** 3 + 0.5 * q ** 4
        outer = 8.0 / 3.0 * q - 3.0 * q ** 2 + 6.0 / 5.0 * q ** 3 - q ** 4 / 6.0 - 1.0 / (15.0 * q ** 2)
        g = np.where(q < 1.0, inner, outer) / q
    g[0] = 4.0 / 3.0
    return g


def _lookup(table, q2):
    f = 10000.0 * q2
    i = f.detach().to(torch.int64).clamp(max=39999)
    t = f - i
    return table[i] * (1.0 - t) + table[i + 1] * t


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _direct_gravity(x, h, m, table):
    """sum_j G m_j (r_j - r_i) g(|r_ij|) with the softened kernel at the mean h, chunked over i."""
    n = len(x)
    out = torch.zeros_like(x)
    step = max(1, (1 << 27) // n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [x[None, :, k] - x[a:b, k, None] for k in range(3)]
        d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        hb = 0.5 * (h[None, :] + h[a:b, None])
        f = d2.clamp(min=1e-300).rsqrt() ** 3
        near = torch.nonzero(d2 < (4.0 - 1e-12) * hb * hb, as_tuple=True)
        hn = hb[near]
        f[near] = _lookup(table, d2[near] / (hn * hn)) / hn ** 3
        f = f * (G * m)[None, :]
        for k in range(3):
            out[a:b, k] = (d[k] * f).sum(1)
    return out


def _pairs(x, h):
    """Ordered pairs (i, j), i != j, with |r_i - r_j| < h_i + h_j."""
    n = len(x)
    ii, jj = [], []
    step = max(1, (1 << 27) // n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d2 = sum((x[a:b, k, None] - x[None, :, k]) ** 2 for k in range(3))
        i, j = torch.nonzero(d2 < (h[a:b, None] + h[None, :]) ** 2, as_tuple=True)
        keep = i + a != j
        ii.append(i[keep] + a)
        jj.append(j[keep])
    return torch.cat(ii), torch.cat(jj)


def _tillotson(rho, u, eos):
    """Pressure and sound speed of the Tillotson equation of state; eos = (a, b, A)."""
    mat = basalt()
    rho0, B, al, be, u0, uiv, ucv = (mat[k] for k in ("rho0", "B", "alpha", "beta", "u0", "uiv", "ucv"))
    a, b, A = eos
    eta = rho / rho0
    mu = eta - 1.0
    w = u / (u0 * eta * eta) + 1.0
    pc = (a + b / w) * rho * u + A * mu + B * mu * mu
    csc = a * u + b * u * (3.0 * w - 2.0) / w ** 2 + A / rho0 + 2.0 * B * mu / rho0 + \
        (a * rho + b * rho / w ** 2) * pc / rho ** 2
    x = rho0 / rho - 1.0
    eb, ea = torch.exp(-torch.clamp(be * x, max=70.0)), torch.exp(-torch.clamp(al * x * x, max=70.0))
    pe = a * rho * u + (b * rho * u / w + A * mu * eb) * ea
    dr = a * u + ea * (b * u * (3.0 * w - 2.0) / w ** 2) + ea * (b * u * rho / w) * rho0 * (2.0 * al * x) / rho ** 2 + \
        ea * A * eb * (1.0 / rho0 + rho0 * mu / rho ** 2 * (2.0 * al * x + be))
    cse = torch.clamp(dr + (a * rho + ea * b * rho / w ** 2) * pe / rho ** 2, min=0.0)
    hot, mid = (rho <= rho0) & (u > ucv), (rho <= rho0) & (u > uiv) & (u <= ucv)
    f = (u - uiv) / (ucv - uiv)
    p = torch.where(hot, pe, torch.where(mid, f * pe + (1.0 - f) * pc, pc))
    cs = torch.where(hot, cse, torch.where(mid, f * cse + (1.0 - f) * csc, csc))
    return p, torch.sqrt(torch.maximum(cs, 0.25 * A / rho0 + 0.0 * cs))


def _gas_evaluate(x, h, v, rho, u, m, eos, table, soft=None):
    """Accelerations, drho, du and the sound speed of the gas terms (pressure, artificial viscosity with
    alpha 1.5 and beta 3, continuity), and the neighbour counts."""
    p, cs = _tillotson(rho, u, eos)
    i, j = _pairs(x.detach(), h)
    d = x[i] - x[j]
    hb = 0.5 * (h[i] + h[j])
    d2 = (d * d).sum(1)
    g = d * (_lookup(table, d2 / (hb * hb)) / hb ** 5)[:, None]
    w = v[j] - v[i]
    wg = (w * g).sum(1)
    dvdr = -(w * d).sum(1)
    mu = hb * dvdr / (d2 + 0.01 * hb * hb)
    av = (-1.5 * 0.5 * (cs[i] + cs[j]) * mu + 3.0 * mu * mu) / (0.5 * (rho[i] + rho[j]))
    av = torch.where(dvdr < 0.0, av, torch.zeros_like(av))
    pr = p / (rho * rho)
    a = torch.zeros_like(x) if soft is None else _direct_gravity(x, h, m, soft)
    a = a.index_add(0, i, -(m[j] * (pr[i] + pr[j] + av))[:, None] * g)
    zero = torch.zeros_like(rho)
    heat = zero.index_add(0, i, -m[j] * 0.5 * av * wg)
    divv = zero.index_add(0, i, m[j] / rho[i] * wg)
    return a, -rho * divv, heat - p / rho * divv, cs, torch.bincount(i, minlength=len(m))


def _density_floor():
    return basalt()["rho_lo"]


def _gas_step(q, h, m, dt, eos, table, soft=None):
    """One predictor-corrector step of q = (x, v, a, rho, drho, u, du); returns q and the Courant step."""
    x, v, a, rho, drho, u, du = q
    x1, v1 = x + v * dt + a * (0.5 * dt * dt), v + a * dt
    r0, e0 = rho + drho * dt, u + du * dt
    floor = _density_floor()
    drho = torch.where((r0 <= floor) & (drho < 0.0), torch.zeros_like(drho), drho)
    du = torch.where((e0 <= 0.0) & (du < 0.0), torch.zeros_like(du), du)
    r1, e1 = torch.clamp(r0, min=floor), torch.clamp(e0, min=0.0)
    a1, drho1, du1, cs, _ = _gas_evaluate(x1, h, v1, r1, e1, m, eos, table, soft)
    x2 = x1 - (a - a1) * (dt * dt / 6.0)
    v2 = v1 - 0.5 * (a - a1) * dt
    r2, e2 = r1 - 0.5 * (drho - drho1) * dt, e1 - 0.5 * (du - du1) * dt
    drho1 = torch.where((r2 <= floor) & (drho1 < 0.0), torch.zeros_like(drho1), drho1)
    du1 = torch.where((e2 <= 0.0) & (du1 < 0.0), torch.zeros_like(du1), du1)
    nxt = min(10.0, float((0.2 * h / cs).min()))
    return (x2, v2, a1, torch.clamp(r2, min=floor), drho1, torch.clamp(e2, min=0.0), du1), nxt


def _gas_tensors(a):
    dev = _device()
    t = {k: torch.tensor(a[k], dtype=torch.float64, device=dev) for k in ("r", "v", "m", "rho", "u")}
    x, h, v = t["r"][:, :3].contiguous(), t["r"][:, 3].contiguous(), t["v"][:, :3].contiguous()
    return x, h, v, t["m"], t["rho"], t["u"]


def exact(case, seed):
    """What `run` returns on a new state.  None for the solid impacts: their damage model decides for each
    particle between no growth and full growth on the last bits of its stress, so that two 64-bit runs may
    differ.  None above a size that takes too long."""
    kind, n = case["kind"], case.get("n", 0)
    dev = _device()
    table = torch.tensor(_m4_table(), device=dev)
    mat = basalt()
    eos = tuple(torch.tensor(mat[k], dtype=torch.float64, device=dev) for k in ("a", "b", "A"))
    if kind == "gas":
        if n * float(n) * case["steps"] > (1e11 if case["gravity"] else 4e11):
            return None
        a = _gas_inputs(case, seed)
        x, h, v, m, rho, u = _gas_tensors(a)
        soft = torch.tensor(_softening_table(), device=dev) if case["gravity"] else None
        z = torch.zeros_like(rho)
        q, dt = (x, v, torch.zeros_like(x), rho, z, u, z), a["dt"]
        for _ in range(case["steps"]):
            q, dt = _gas_step(q, h, m, dt, eos, table, soft)
        lane = torch.zeros_like(h)[:, None]
        return dict(r=torch.cat([q[0], h[:, None]], 1), v=torch.cat([q[1], lane], 1), rho=q[3], u=q[5])
    if kind == "evaluate":
        if n > 600000:
            return None
        x, h, v, m, rho, u = _gas_tensors(_gas_inputs(dict(case, bodies=2), seed))
        acc, drho, du, _, cnt = _gas_evaluate(x, h, v, rho, u, m, eos, table)
        return dict(dv=torch.cat([acc, torch.zeros_like(h)[:, None]], 1), drho=drho, du=du, ncnt=None)
    if kind == "adjoint":
        if n * case["steps"] > 400000:
            return None
        a = _gas_inputs(dict(case, bodies=2), seed)
        x, h, v, m, rho, u = _gas_tensors(a)
        leaves = [t.clone().requires_grad_() for t in (x, v, rho, u, *eos)]
        z = torch.zeros_like(rho)
        q = (leaves[0], leaves[1], torch.zeros_like(x), leaves[2], z, leaves[3], z)
        for _ in range(case["steps"]):
            q, _ = _gas_step(q, h, m, a["dt"], leaves[4:], table)
        sr, sv, su = (torch.tensor(s, device=dev) for s in _objective(a))
        J = (q[0] * sr).sum() + (q[1] * sv).sum() + (q[5] * su).sum()
        g = torch.autograd.grad(J, leaves)
        return dict(r=g[0], v=g[1], rho=g[2], u=g[3], eos=torch.stack(g[4:])[None, :])
    if kind in ("nbody", "direct"):
        if n * float(n) * case.get("steps", 1) > 2e11:
            return None
        r, v, m = _nbody_inputs(case, seed)
        if kind == "direct":
            r[:, 3] = 2.0e3
        r, v, m = (torch.tensor(t, device=dev) for t in (r, v, m))
        soft = torch.tensor(_softening_table(), device=dev)
        h = r[:, 3].contiguous()
        if kind == "direct":
            return dict(dv=_direct_gravity(r[:, :3].contiguous(), h, m, soft))
        for _ in range(case["steps"]):
            r = r + v * (0.5 * NBODY_DT)
            v[:, :3] += _direct_gravity(r[:, :3].contiguous(), h, m, soft) * NBODY_DT
            r = r + v * (0.5 * NBODY_DT)
        return dict(r=r, v=v)
    return None
