"""Timed workloads of the MD engine, through its public Python entry points.

What the listed cases stand for (sizes are those of the repository's own
configurations, tests and benchmark, or generic ones of the same range):

  argon_256           the smallest replica of the batched workload: a step is
                      a handful of launches, so latency is what counts
  argon_10000         liquid argon, plain velocity Verlet (the LJ-only path)
  water_267           the smallest water replica under Langevin dynamics
  water_7938          a large water replica (still one-workgroup binning)
  water_24576         the 8,192-molecule box, Nose-Hoover, default skin
  water_52773_order5  an odd molecule count, mixed-radix grid, order 5
  water_196608_npt    the headline box: SETTLE, Nose-Hoover, C-rescale
  polymer_10000       200 chains x 50 beads, every bond SHAKE-constrained
  batch_32            32 uneven argon and water replicas, one graph per step
  frames_water_24576  energies and forces of new configurations (a rerun over
                      trajectory frames: every frame rebuilds the list)
  frames_tilted       the same for a sheared cell, order 5, odd grid, switched
                      LJ (the general pair loop)
  predictor_train     the SHAKE predictor trained on logged rows, then used

A dynamics pass advances the state by ``steps`` steps and reads back the
frame (positions, velocities, energies), as a program that writes a
trajectory does; the next pass goes on from there.  Inputs come from the
seed alone: tetrahedral water (a proton-ordered diamond lattice with thermal
displacements, at 1 g/cm^3), fcc argon with thermal displacements at the
liquid's density, extended polymer chains, Maxwell-Boltzmann velocities.
Pair counts, charges and forces are those of the condensed phase.

``exact`` restates every workload but the stochastic barostat in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from heddlemd_amd import systems
from heddlemd_amd import units as U
from heddlemd_amd.engine import Batch, ShakePredictor, engine_for

NM = U.length(1e-9)
FS = U.time(1e-15)
M_WATER_KG = systems.M_O_KG + 2 * systems.M_H_KG
SIDES = (32, 36, 40, 48, 50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128)


# ---- cases ---------------------------------------------------------------

def _md(name, system, n, integrator, steps, **more):
    return dict(name=name, kind="md", system=system, n=n, integrator=integrator, steps=steps,
                **more)


def listed():
    return [
        _md("argon_256", "argon", 256, "langevin", 100, skin_nm=0.0),
        _md("argon_10000", "argon", 10000, "nve", 50, skin_nm=0.0),
        _md("water_267", "water", 89, "langevin", 50, skin_nm=0.0, order=4),
        _md("water_7938", "water", 2646, "langevin", 50, skin_nm=0.0, order=4),
        _md("water_24576", "water", 8192, "nvt", 50, skin_nm=0.0, order=4, grid=64),
        _md("water_52773_order5", "water", 17591, "nvt", 40, skin_nm=0.2, order=5),
        _md("water_196608_npt", "water", 65536, "npt", 50, skin_nm=0.14, order=4, grid=128),
        dict(name="polymer_10000", kind="md", system="polymer", n=200, beads=50,
             integrator="nvt", steps=50, skin_nm=0.0),
        dict(name="batch_32", kind="batch", replicas=32, steps=20),
        dict(name="frames_water_24576", kind="frames", n=8192, frames=4, skin_nm=0.0, order=4,
             tilt=0.0, switch=False),
        dict(name="frames_tilted", kind="frames", n=4001, frames=4, skin_nm=0.1, order=5,
             tilt=0.12, switch=True),
        dict(name="predictor_train", kind="train", rows=200_003, batch=4096, epochs=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["argon", "water", "water", "water", "polymer", "batch", "frames",
                       "frames", "train"])
    skin = rng.choice([0.0, 0.1, 0.14, 0.2])
    if kind == "argon":
        return dict(kind="md", system="argon", n=_log_int(rng, 256, 40000),
                    integrator=rng.choice(["nve", "langevin"]), steps=rng.randrange(20, 60),
                    skin_nm=skin)
    if kind == "water":
        n = _log_int(rng, 89, 50000)
        return dict(kind="md", system="water", n=n,
                    integrator=rng.choice(["nvt", "npt", "langevin"]),
                    steps=rng.randrange(20, 50), skin_nm=skin, order=rng.choice([4, 4, 5]))
    if kind == "polymer":
        return dict(kind="md", system="polymer", n=rng.randrange(40, 300),
                    beads=rng.randrange(24, 60), integrator="nvt", steps=rng.randrange(20, 60),
                    skin_nm=skin)
    if kind == "batch":
        return dict(kind="batch", replicas=rng.randrange(8, 33), steps=rng.randrange(10, 25))
    if kind == "frames":
        return dict(kind="frames", n=_log_int(rng, 120, 30000), frames=rng.randrange(2, 5),
                    skin_nm=skin, order=rng.choice([4, 5]), tilt=rng.choice([0.0, 0.0, 0.08]),
                    switch=rng.random() < 0.3)
    return dict(kind="train", rows=_log_int(rng, 20000, 250000),
                batch=rng.choice([1024, 4096, 16384]), epochs=rng.randrange(1, 3))


# ---- inputs --------------------------------------------------------------

def _cells(n_cells):
    """Near-cubic (mx, my, mz) with at least n_cells cells and few left over."""
    m0 = max(int(n_cells ** (1.0 / 3.0)), 1)
    best = None
    for mx in range(max(m0 - 1, 1), m0 + 2):
        for my in range(mx, m0 + 3):
            mz = max(-(-n_cells // (mx * my)), my)
            cost = mx * my * mz / n_cells + 0.15 * (mz / mx - 1.0)
            if best is None or cost < best[0]:
                best = (cost, (mx, my, mz))
    return best[1]


def _sites(rng, cells, basis, n):
    """n of the basis' sites over the cells, as fractional coordinates and
    the index of the basis site."""
    mx, my, mz = cells
    g = np.stack(np.meshgrid(np.arange(mx), np.arange(my), np.arange(mz), indexing="ij"), -1)
    f = (g.reshape(-1, 1, 3) + basis[None]).reshape(-1, 3) / np.array(cells, np.float64)
    which = np.tile(np.arange(len(basis)), mx * my * mz)
    keep = np.sort(rng.permutation(len(f))[:n])
    return f[keep] - 0.5, which[keep]


FCC = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]], np.float64)


def _rotate(v, w):
    """Rows of v rotated by the rotation vectors w."""
    a = np.linalg.norm(w, axis=1, keepdims=True)
    k = w / np.maximum(a, 1e-12)
    return (v * np.cos(a) + np.cross(k, v) * np.sin(a)
            + k * np.sum(k * v, axis=1, keepdims=True) * (1 - np.cos(a)))


def _box(lengths, tilt):
    L = [systems.box_length(x) for x in lengths]
    t = [float(np.float32(tilt * L[0])), float(np.float32(-0.6 * tilt * L[0])),
         float(np.float32(0.8 * tilt * L[1]))]
    return np.array(L + t)


def _cell(lattice):
    lx, ly, lz, xy, xz, yz = (float(v) for v in lattice)
    return np.array([[lx, xy, xz], [0.0, ly, yz], [0.0, 0.0, lz]])


def _wrap(x, lattice):
    H = _cell(lattice)
    f = x @ np.linalg.inv(H).T
    return x - np.floor(f + 0.5) @ H.T


def _cutoff(want_nm, lattice, skin_nm):
    """The cutoff (Bohr) and skin (Bohr or None for the default), capped as
    the replica workload caps them: cutoff + skin within 0.45 box widths."""
    H = _cell(lattice)
    width = 1.0 / np.linalg.norm(np.linalg.inv(H), axis=1).max()
    rc = min(want_nm * NM, 0.45 * width / 1.3)
    return rc, (None if skin_nm == 0.0 else min(skin_nm * NM, 0.3 * rc))


def _table(types, cutoff, pairs, switch=False):
    sig, eps = np.zeros((types, types)), np.zeros((types, types))
    for (a, b), (s, e) in pairs.items():
        sig[a, b] = sig[b, a] = s
        eps[a, b] = eps[b, a] = e
    cut = np.full((types, types), cutoff)
    return systems.LJTable(types, sig, eps, cut, 0.85 * cut if switch else cut.copy())


def _argon(case, rng):
    n = case["n"]
    cells = _cells(-(-n // 4))
    f, _ = _sites(rng, cells, FCC, n)
    a = (n / 2.1e28 / (cells[0] * cells[1] * cells[2])) ** (1 / 3) * 1e9 * NM
    lattice = _box(np.array(cells) * a, 0.0)
    x = _wrap(f * lattice[:3] + rng.normal(scale=0.012 * NM, size=(n, 3)), lattice)
    rc, skin = _cutoff(0.85, lattice, case["skin_nm"])
    posq = np.zeros((n, 4), np.float32)
    posq[:, :3] = x
    s = systems.System(
        name="argon", posq=posq, mass=np.full(n, U.mass(6.6335e-26), np.float32),
        types=np.zeros(n, np.uint32), lattice=lattice,
        lj=_table(1, rc, {(0, 0): (U.length(3.405e-10), U.energy(1.654e-21))}))
    return s, skin


def _water_frames(case, rng, frames, tilt):
    """The box and `frames` independent thermal configurations of it."""
    n = case["n"]
    cells = _cells(-(-n // 8))
    basis = np.concatenate([FCC, FCC + 0.25])
    f, which = _sites(rng, cells, basis, n)
    volume = n * M_WATER_KG / 1000.0
    a = (volume / (cells[0] * cells[1] * cells[2])) ** (1 / 3) * 1e9 * NM
    lattice = _box(np.array(cells) * a, tilt)
    H = _cell(lattice)
    # the four bond directions of a tetrahedral site: sites of the first
    # sublattice donate along two of them, the second's along the other two
    d = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]]) / math.sqrt(3.0)
    donors = np.stack([d[0], d[1]]), np.stack([-d[2], -d[3]])
    second = which >= 4
    h1 = np.where(second[:, None], donors[1][0], donors[0][0])
    h2 = np.where(second[:, None], donors[1][1], donors[0][1])
    # the molecule's own geometry along those directions: exactly d_OH long
    # and 109.47 degrees apart
    th = math.radians(109.47)
    mid = (h1 + h2) / np.linalg.norm(h1 + h2, axis=1, keepdims=True)
    per = (h1 - h2) / np.linalg.norm(h1 - h2, axis=1, keepdims=True)
    d_oh = U.length(1.0e-10)
    h1 = d_oh * (math.cos(th / 2) * mid + math.sin(th / 2) * per)
    h2 = d_oh * (math.cos(th / 2) * mid - math.sin(th / 2) * per)
    out = []
    for _ in range(frames):
        # frames far apart: atoms have moved by more than any skin
        o = (f @ H.T + rng.uniform(-0.4, 0.4, 3) * NM
             + rng.normal(scale=0.009 * NM, size=(n, 3)))
        w = rng.normal(scale=0.1, size=(n, 3))
        x = np.stack([o, o + _rotate(h1, w), o + _rotate(h2, w)], axis=1).reshape(-1, 3)
        posq = np.empty((3 * n, 4), np.float32)
        posq[:, :3] = _wrap(x, lattice)
        posq[:, 3] = np.tile(np.array([-0.82, 0.41, 0.41], np.float32), n)
        out.append(posq)
    return lattice, out


def _water(case, rng, frames=1):
    lattice, posqs = _water_frames(case, rng, frames, case.get("tilt", 0.0))
    n = case["n"]
    rc, skin = _cutoff(0.9, lattice, case["skin_nm"])
    grid = tuple(case.get("grid") or min(SIDES, key=lambda g: abs(math.log(g * 0.1 * NM / L)))
                 for L in (float(v) for v in lattice[:3]))
    lj = _table(2, rc, {(0, 0): (U.length(0.3166e-9), U.energy(650.0 / U.AVOGADRO)),
                        (0, 1): (U.length(1e-10), 0.0), (1, 1): (U.length(1e-10), 0.0)},
                case.get("switch", False))
    d_oh = U.length(1.0e-10)
    m_o, m_h = U.mass(systems.M_O_KG), U.mass(systems.M_H_KG)
    s = systems.System(
        name="water", posq=posqs[0], mass=np.tile(np.array([m_o, m_h, m_h], np.float32), n),
        types=np.tile(np.array([0, 1, 1], np.uint32), n), lattice=lattice, lj=lj,
        spme=systems.SpmeParams(systems.ewald_alpha(rc, 1e-5), rc, grid, case.get("order", 4)),
        water_groups=np.arange(3 * n, dtype=np.uint32).reshape(n, 3),
        water_geom=(d_oh, 2.0 * d_oh * math.sin(math.radians(109.47) / 2)),
        excl_key=np.repeat(np.arange(n, dtype=np.uint32), 3))
    return s, skin, posqs


def _polymer(case, rng):
    """Extended chains side by side along z, each turned about its axis and
    shifted along it; bonds and angles at their equilibrium values."""
    nc, nb = case["n"], case["beads"]
    bond, half = 0.153 * NM, math.radians(57.0)
    lz = nb * bond * math.sin(half) + 0.3 * NM
    m = U.mass(14.0 * U.AMU_TO_KG)
    volume = nc * nb * 14.0 * U.AMU_TO_KG / 800.0 * 1e27 * NM ** 3
    nx = max(int(round(math.sqrt(nc))), 1)
    ny = -(-nc // nx)
    side = math.sqrt(volume / lz / (nx * ny))
    lattice = _box([nx * side, ny * side, lz], 0.0)
    k = np.arange(nb)
    phi = rng.uniform(0, 2 * math.pi, nc)
    off = 0.5 * bond * math.cos(half) * np.where(k % 2 == 0, 1.0, -1.0)
    c = np.arange(nc)
    x = np.empty((nc, nb, 3))
    x[..., 0] = ((c % nx) * side)[:, None] + np.cos(phi)[:, None] * off
    x[..., 1] = ((c // nx) * side)[:, None] + np.sin(phi)[:, None] * off
    x[..., 2] = rng.uniform(0, lz, nc)[:, None] + k * bond * math.sin(half)
    n = nc * nb
    posq = np.zeros((n, 4), np.float32)
    posq[:, :3] = _wrap(x.reshape(-1, 3), lattice)
    rc, skin = _cutoff(1.0, lattice, case["skin_nm"])
    first = np.arange(nc)[:, None] * nb + np.arange(nb - 2)
    ijk = np.stack([first, first + 1, first + 2], -1).reshape(-1, 3).astype(np.uint32)
    s = systems.System(
        name="polymer", posq=posq, mass=np.full(n, m, np.float32),
        types=np.zeros(n, np.uint32), lattice=lattice,
        lj=_table(1, rc, {(0, 0): (U.length(0.395e-9), U.energy(382.0 / U.AVOGADRO))}),
        excl_key=(np.repeat(np.arange(nc), nb) * 64 + np.tile(np.arange(nb), nc)).astype(np.uint32),
        excl_span=2,
        shake_groups=[(list(range(g * nb, g * nb + nb)), [(b, b + 1, bond) for b in range(nb - 1)])
                      for g in range(nc)],
        angles=(ijk, np.full(len(ijk), U.energy(520e3 / U.AVOGADRO)),
                np.full(len(ijk), 2 * half)))
    return s, skin


def _velocities(rng, mass, kt):
    m = mass.astype(np.float64)
    v = rng.normal(size=(3, len(m))) * np.sqrt(kt / m)
    return (v - (v * m).sum(1, keepdims=True) / m.sum()).astype(np.float32)


def _temperature(case):
    return U.temperature({"argon": 300.0 if case["integrator"] == "langevin" else 94.0,
                          "water": 300.0, "polymer": 400.0}[case["system"]])


def _md_inputs(case, seed):
    rng = np.random.default_rng([seed, case["n"]])
    if case["system"] == "argon":
        s, skin = _argon(case, rng)
    elif case["system"] == "water":
        s, skin, _ = _water(case, rng)
    else:
        s, skin = _polymer(case, rng)
    return s, skin, _velocities(rng, s.mass, _temperature(case))


def _md_engine(case, seed):
    s, skin, v = _md_inputs(case, seed)
    kt = _temperature(case)
    how = case["integrator"]
    more = {}
    if how == "langevin":
        more["langevin"] = dict(friction=1.0 / U.time(1e-12), kt=kt, seed=17)
    if how in ("nvt", "npt"):
        more.update(nhc_kt=kt, nhc_tau=100 * FS)
    if how == "npt":
        more["crescale"] = dict(pressure=U.pressure(1e5), tau=U.time(1e-12),
                                compressibility=U.inv_pressure(4.5e-10), kt=kt, seed=13)
    e = engine_for(s, dt=2 * FS, velocities=v, r_skin=skin, **more)
    if case["system"] == "polymer":
        e.set_shake_tolerance(5e-5, 1e-8, 500)
    if s.n_constraints:
        e.constrain_velocities()
    return e


def _replicas(case):
    """Half argon, half water, atom counts log-uniform in 256..8192 (the
    counts belong to the case; each replica's state is made from the seed)."""
    rng = np.random.default_rng([case["replicas"], 5])
    out = []
    for r in range(case["replicas"]):
        n = int(round(math.exp(rng.uniform(math.log(256), math.log(8192)))))
        kind = "argon" if 2 * r < case["replicas"] else "water"
        out.append(dict(kind="md", system=kind, n=n if kind == "argon" else max(n // 3, 89),
                        integrator="langevin", steps=case["steps"], skin_nm=0.0, order=4))
    return out


def _train_inputs(case, seed):
    """Rows as the SHAKE log holds them: first-order multipliers of the
    constraint and its neighbours (1e-3), couplings near -0.3, the strain;
    the target solves the coupled system to second order."""
    rng = np.random.default_rng([seed, case["rows"]])
    n = case["rows"]
    x = rng.normal(scale=1.2e-3, size=(n, 8))
    x[:, 5:7] = rng.normal(-0.3, 0.06, size=(n, 2))
    t = (x[:, 0] - x[:, 5] * x[:, 1] - x[:, 6] * x[:, 2] + 0.09 * x[:, 4]
         + 0.4 * x[:, 0] * x[:, 7] / 1.2e-3 * 0.1 + rng.normal(scale=5e-5, size=n))
    p = np.zeros(8 * 64 + 64 + 64 * 64 + 64 + 64 + 2)
    p[:512] = rng.uniform(-1, 1, 512) / math.sqrt(8)
    p[576:576 + 4096] = rng.uniform(-1, 1, 4096) / 8.0
    p[4736:4800] = rng.uniform(-1, 1, 64) * 0.05
    return x.astype(np.float32), t.astype(np.float32), p.astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "md":
        return dict(case=case, engine=_md_engine(case, seed))
    if case["kind"] == "batch":
        engines = [_md_engine(c, seed + 31 * r) for r, c in enumerate(_replicas(case))]
        return dict(case=case, engines=engines, batch=Batch(engines))
    if case["kind"] == "frames":
        rng = np.random.default_rng([seed, case["n"]])
        s, skin, posqs = _water(case, rng, case["frames"])
        return dict(case=case, engine=engine_for(s, r_skin=skin), posqs=posqs)
    x, t, p = _train_inputs(case, seed)
    return dict(case=case, model=ShakePredictor(seed=1), x=x, t=t, p=p)


# ---- passes --------------------------------------------------------------

def _frame(e):
    """One trajectory frame: unwrapped positions, velocities, energies."""
    posq, image = e.positions(images=True)
    sc = e.scalars()
    return dict(x=posq[:, :3] + image.T * e.lattice()[:3].astype(np.float32),
                v=e.velocities(), energy=np.array([sc["ke"], sc["pe"]]))


def run(state):
    case = state["case"]
    if case["kind"] == "md":
        e = state["engine"]
        e.step(case["steps"], scalars_last=True)
        return _frame(e)
    if case["kind"] == "batch":
        state["batch"].step(case["steps"], scalars_last=True)
        frames = [_frame(e) for e in state["engines"]]
        return dict(x=np.concatenate([f["x"] for f in frames]),
                    v=np.concatenate([f["v"] for f in frames], axis=1),
                    energy=np.stack([f["energy"] for f in frames]))
    if case["kind"] == "frames":
        e, out = state["engine"], []
        for posq in state["posqs"]:
            e.set_positions(posq)
            e.force_eval(scalars=True)
            pe, _ = e.per_atom()
            sc = e.scalars()
            out.append(dict(f=e.forces(), pe=pe,
                            energy=np.array([sc["pe"], sc["e_recip"]]),
                            virial=np.array([sc["virial"], sc["w_recip"]])))
        return out
    m = state["model"]
    m.params = state["p"]
    loss = m.train(state["x"], state["t"], epochs=case["epochs"], batch=case["batch"], lr=2e-3,
                   seed=7)
    return dict(params=m.params, loss=loss, nu=m.predict(state["x"]))


# ---- the least work of a pass ---------------------------------------------

def _eval_work(atoms, water, order):
    """One force evaluation: every pair within the cutoff once (55 flops with
    the real-space Ewald term, 20 without), the transforms there and back,
    spreading and gathering; positions in, forces out."""
    rc = 0.9 if water else 0.85
    density = (1e-27 * 1000.0 / M_WATER_KG * 3) if water else 21.0
    flops = (55.0 if water else 20.0) * atoms * density * 4.18879 * rc ** 3 / 2
    if water:
        grid = atoms / density * 1000.0
        flops += 2 * 2.5 * grid * math.log2(grid) + atoms * order ** 3 * 11
    return dict(bytes=28.0 * atoms, flops=flops)


def _step_work(case):
    atoms = case["n"] * {"argon": 1, "water": 3, "polymer": case.get("beads", 1)}[case["system"]]
    w = _eval_work(atoms, case["system"] == "water", case.get("order", 4))
    return dict(bytes=case["steps"] * (w["bytes"] + 56.0 * atoms),
                flops=case["steps"] * w["flops"])


def work(case):
    if case["kind"] == "md":
        return _step_work(case)
    if case["kind"] == "batch":
        # the mean of the counts' distribution, 2286 atoms
        half = case["replicas"] / 2
        a = _step_work(dict(system="argon", n=2286 * half, steps=case["steps"]))
        w = _step_work(dict(system="water", n=762 * half, steps=case["steps"]))
        return {k: a[k] + w[k] for k in a}
    if case["kind"] == "frames":
        w = _eval_work(3 * case["n"], True, case["order"])
        return {k: case["frames"] * w[k] for k in w}
    rows = case["rows"]
    return dict(bytes=rows * 36.0 * (case["epochs"] + 1),
                flops=rows * 4800.0 * (6 * case["epochs"] + 2))


def tolerance(case):
    # Four times what another order of the 32-bit sums gives.  Dynamics: the
    # rounding of one step travels through the following ones; SHAKE stops at
    # a tolerance (5e-5 Bohr^2), so the chains' velocities agree less well.
    if case["kind"] == "md":
        if case["system"] == "polymer":
            return {"rel": 2e-3, "max": 0.2}
        return {"rel": 2e-4, "max": 2e-2}
    if case["kind"] == "batch":
        return {"rel": 2e-4, "max": 2e-2}
    if case["kind"] == "frames":
        return {"rel": 5e-6, "max": 2e-4}
    return {"rel": 1e-4, "max": 1e-2}


# ---- the same in 64 bits ---------------------------------------------------

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.asarray(a), device=DEV).to(torch.float64)


def _min_image(d, lattice):
    lx, ly, lz, xy, xz, yz = (float(v) for v in lattice)
    c = torch.floor(d[..., 2] / lz + 0.5)
    y = d[..., 1] - c * yz
    b = torch.floor(y / ly + 0.5)
    x = d[..., 0] - c * xz - b * xy
    a = torch.floor(x / lx + 0.5)
    return torch.stack([x - a * lx, y - b * ly, d[..., 2] - c * lz], -1)


class _Field:
    """The force field of a system: pair terms, reciprocal sum, angles."""

    def __init__(self, s):
        self.s, self.n = s, s.posq.shape[0]
        self.q = _t(s.posq[:, 3])
        self.types = torch.as_tensor(s.types.astype(np.int64), device=DEV)
        key = s.excl_key if s.excl_key is not None else np.arange(self.n)
        self.key = torch.as_tensor(np.asarray(key).astype(np.int64), device=DEV)
        self.lattice = [float(np.float32(v)) for v in s.lattice]
        self.sig, self.eps, self.cut, self.rsw = (_t(getattr(s.lj, k)) for k in
                                                  ("sigma", "epsilon", "cutoff", "r_switch"))
        self.rmax = max(float(s.lj.cutoff.max()), s.spme.r_cut if s.spme else 0.0)

    def pairs(self, x):
        """Forces, per-atom energies and the virial of the pair terms."""
        n, lz = self.n, self.lattice[2]
        f = torch.zeros(n, 3, dtype=torch.float64, device=DEV)
        pe = torch.zeros(n, dtype=torch.float64, device=DEV)
        w = torch.zeros((), dtype=torch.float64, device=DEV)
        order = torch.argsort(x[:, 2] - lz * torch.floor(x[:, 2] / lz + 0.5))
        rows = max(min(n, int(3e7 / n)), 64)
        for at in range(0, n, rows):
            i = order[at:at + rows]
            # the slab of atoms that can reach the chunk's z range
            z = x[i, 2] - lz * torch.floor(x[i, 2] / lz + 0.5)
            mid, half = float(z.max() + z.min()) / 2, float(z.max() - z.min()) / 2
            dz = x[:, 2] - mid
            dz = (dz - lz * torch.floor(dz / lz + 0.5)).abs()
            j = torch.nonzero(dz <= half + self.rmax + 1e-6)[:, 0]
            d = _min_image(x[i][:, None] - x[j][None], self.lattice)
            near = ((d * d).sum(-1) <= self.rmax ** 2) & \
                ((self.key[i][:, None] - self.key[j][None]).abs() > self.s.excl_span)
            a, b = torch.nonzero(near, as_tuple=True)
            d, a, b = d[a, b], i[a], j[b]
            r2 = (d * d).sum(-1)
            factor, energy = self._pair_terms(r2, a, b)
            f.index_add_(0, a, factor[:, None] * d)
            pe.index_add_(0, a, 0.5 * energy)
            w += 0.5 * (factor * r2).sum()
        return f, pe, w

    def _pair_terms(self, r2, a, b):
        ta, tb = self.types[a], self.types[b]
        eps, cut, rsw = self.eps[ta, tb], self.cut[ta, tb], self.rsw[ta, tb]
        s6 = (self.sig[ta, tb] ** 2 / r2) ** 3
        e = 4 * eps * (s6 * s6 - s6)
        g = 24 * eps * (2 * s6 * s6 - s6) / r2
        delta = torch.clamp(cut ** 2 - rsw ** 2, min=1e-300)
        tau = torch.where(cut > rsw, torch.clamp((r2 - rsw ** 2) / delta, min=0.0), 0.0 * r2)
        sw = (1 - tau) ** 2 * (1 + 2 * tau)
        g = sw * g + torch.where(cut > rsw, 12 * tau * (1 - tau) / delta, 0.0 * r2) * e
        on = (r2 <= cut ** 2) & (eps != 0)
        factor, energy = torch.where(on, g, 0.0 * r2), torch.where(on, sw * e, 0.0 * r2)
        if self.s.spme is not None:
            al, r = self.s.spme.alpha, torch.sqrt(r2)
            qq = self.q[a] * self.q[b]
            er = torch.erfc(al * r) / r
            on = r <= self.s.spme.r_cut
            energy = energy + torch.where(on, qq * er, 0.0 * r2)
            factor = factor + torch.where(on, qq * (er + 2 * al / math.sqrt(math.pi)
                                                    * torch.exp(-(al * r) ** 2)) / r2, 0.0 * r2)
        return factor, energy

    def recip(self, x):
        """Smooth particle mesh Ewald (Essmann et al. 1995): forces, per-atom
        energies without the self term, total energy and virial."""
        sp, order = self.s.spme, self.s.spme.order
        H = _cell(self.lattice)
        Hi = _t(np.linalg.inv(H))
        dims = torch.tensor(sp.grid, device=DEV)
        fr = x @ Hi.T
        u = (fr - torch.floor(fr + 0.5) + 0.5) * dims
        base = torch.floor(u)
        t = u - base
        w, dw = [], []
        for d in range(order):
            w.append(_bspline(order, t + d))
            dw.append(_bspline(order - 1, t + d) - _bspline(order - 1, t + d - 1))
        w, dw = torch.stack(w, 1), torch.stack(dw, 1)          # (n, order, 3)
        cell = (base.long()[:, None] - torch.arange(order, device=DEV)[None, :, None]) % dims
        rho = torch.zeros(sp.grid, dtype=torch.float64, device=DEV)
        na, nb, nc = sp.grid
        idx = ((cell[:, :, None, None, 0] * nb + cell[:, None, :, None, 1]) * nc
               + cell[:, None, None, :, 2])
        val = (w[:, :, None, None, 0] * w[:, None, :, None, 1] * w[:, None, None, :, 2]
               * self.q[:, None, None, None])
        rho.view(-1).index_add_(0, idx.reshape(-1), val.reshape(-1))
        m = [torch.fft.fftfreq(g, 1.0 / g, dtype=torch.float64, device=DEV) for g in (na, nb)]
        m.append(torch.arange(nc // 2 + 1, dtype=torch.float64, device=DEV))
        k = 2 * math.pi * torch.stack(torch.meshgrid(*m, indexing="ij"), -1) @ Hi
        k2 = (k * k).sum(-1)
        al = sp.alpha
        G = 4 * math.pi / k2 * torch.exp(-k2 / (4 * al * al)) / float(np.linalg.det(H))
        for axis, g in enumerate(sp.grid):
            b = _b_factors(g, order)[: G.shape[axis]]
            G = G * b.view([-1 if a == axis else 1 for a in range(3)])
        G[0, 0, 0] = 0.0
        R = torch.fft.rfftn(rho)
        P = G * (R.real ** 2 + R.imag ** 2)
        hw = torch.full((nc // 2 + 1,), 2.0, dtype=torch.float64, device=DEV)
        hw[0] = hw[-1] = 1.0
        e = 0.5 * (P * hw).sum()
        wv = 0.5 * (P * hw * (1 - k2 / (2 * al * al))).sum()
        V = torch.fft.irfftn(G * R, s=sp.grid, norm="forward").reshape(-1)[idx]
        phi = torch.einsum("nabc,na,nb,nc->n", V, w[..., 0], w[..., 1], w[..., 2])
        g = torch.stack([torch.einsum("nabc,na,nb,nc->n", V, dw[..., 0], w[..., 1], w[..., 2]),
                         torch.einsum("nabc,na,nb,nc->n", V, w[..., 0], dw[..., 1], w[..., 2]),
                         torch.einsum("nabc,na,nb,nc->n", V, w[..., 0], w[..., 1], dw[..., 2])], 1)
        return -self.q[:, None] * ((g * dims) @ Hi), 0.5 * self.q * phi, e, wv

    def angles(self, x):
        ijk, kth, th0 = self.s.angles
        i, j, k = (torch.as_tensor(ijk[:, c].astype(np.int64), device=DEV) for c in range(3))
        a, b = _min_image(x[i] - x[j], self.lattice), _min_image(x[k] - x[j], self.lattice)
        la, lb = a.norm(dim=1), b.norm(dim=1)
        sn, cs = torch.linalg.cross(a, b).norm(dim=1) / (la * lb), (a * b).sum(1) / (la * lb)
        th = torch.atan2(sn, cs) - _t(th0)
        g = -_t(kth) * th / sn
        fi = g[:, None] * (cs[:, None] * a / la[:, None] ** 2 - b / (la * lb)[:, None])
        fk = g[:, None] * (cs[:, None] * b / lb[:, None] ** 2 - a / (la * lb)[:, None])
        f = torch.zeros_like(x)
        f.index_add_(0, i, fi)
        f.index_add_(0, k, fk)
        f.index_add_(0, j, -fi - fk)
        return f, 0.5 * (_t(kth) * th * th).sum()

    def all(self, x):
        """Forces, per-atom energies, (energy, reciprocal energy), (virial,
        reciprocal virial)."""
        f, pe, w = self.pairs(x)
        e, er, wr = pe.sum(), 0.0, 0.0
        if self.s.spme is not None:
            g, per, er, wr = self.recip(x)
            own = self.s.spme.alpha / math.sqrt(math.pi) * self.q ** 2
            f, pe = f + g, pe + per - own
            e = pe.sum()
        if self.s.angles is not None:
            g, ea = self.angles(x)
            f, e = f + g, e + ea
        return f, pe, (e, er), (w + wr, wr)


def _bspline(order, x):
    v = [((x - i >= 0) & (x - i < 1)).to(torch.float64) for i in range(order)]
    for o in range(2, order + 1):
        v = [(x - i) / (o - 1) * v[i] + (o - x + i) / (o - 1) * v[i + 1]
             for i in range(order - o + 1)]
    return v[0]


def _b_factors(n, order):
    m = [float(_bspline(order, torch.tensor(float(j), dtype=torch.float64)))
         for j in range(1, order)]
    k = np.arange(n)
    s = np.abs(sum(v * np.exp(2j * np.pi * k * j / n) for j, v in enumerate(m))) ** 2
    small = s < 1e-7
    s = np.where(small, 0.5 * (np.roll(s, 1) + np.roll(s, -1)), s)
    return _t(1.0 / s)


class _Constraints:
    """Distance constraints of equal groups: positions moved along the bonds
    of the step's start (Newton on the multipliers), bond-relative velocities
    removed (one linear solve)."""

    def __init__(self, s):
        if s.water_groups is not None:
            a, b = s.water_geom
            self.atoms = torch.as_tensor(s.water_groups.astype(np.int64), device=DEV)
            ij, d = [(0, 1), (0, 2), (1, 2)], [a, a, b]
        else:
            self.atoms = torch.as_tensor(np.array([g[0] for g in s.shake_groups]), device=DEV)
            ij, d = [c[:2] for c in s.shake_groups[0][1]], [c[2] for c in s.shake_groups[0][1]]
        self.i, self.j = (torch.tensor([c[k] for c in ij], device=DEV) for k in (0, 1))
        self.d2 = _t(d) ** 2
        E = np.zeros((len(ij), self.atoms.shape[1]))
        for c, (a, b) in enumerate(ij):
            E[c, a], E[c, b] = 1.0, -1.0
        im = 1.0 / s.mass[np.asarray(self.atoms[0].cpu())].astype(np.float64)
        self.im = _t(im)
        self.E = _t(E)
        self.K = _t((E * im) @ E.T)                 # (C, C) coupling of the constraints
        self.L = [float(np.float32(v)) for v in s.lattice]

    def bonds(self, x):
        g = x[self.atoms]
        return _min_image(g[:, self.i] - g[:, self.j], self.L)

    def _solve(self, A, b):
        return torch.linalg.solve(A.cpu(), b.cpu()).to(DEV)

    def _spread(self, lam, g):
        return torch.matmul(self.E.T, lam[..., None] * g) * self.im[:, None]

    def positions(self, x, old):
        """The correction of every atom."""
        g, u = self.bonds(old), self.bonds(x)
        lam = torch.zeros(u.shape[:2], dtype=torch.float64, device=DEV)
        r = u
        for _ in range(30):
            res = (r * r).sum(-1) - self.d2
            if float((res / self.d2).abs().max()) < 1e-14:
                break
            J = 2 * self.K * torch.matmul(r, g.transpose(1, 2).contiguous())
            lam = lam - self._solve(J, res)
            r = u + torch.matmul(self.K, lam[..., None] * g)
        out = torch.zeros_like(x)
        out[self.atoms] = self._spread(lam, g)
        return out

    def velocities(self, x, v):
        r = self.bonds(x)
        vv = v[self.atoms]
        rel = (r * (vv[:, self.i] - vv[:, self.j])).sum(-1)
        A = self.K * torch.matmul(r, r.transpose(1, 2).contiguous())
        out = torch.zeros_like(v)
        out[self.atoms] = self._spread(-self._solve(A, rel), r)
        return out


def _philox_normal(seed, counter, n, axis):
    """Philox4x32-10 (Salmon et al., SC11), Box-Muller of the first two words
    of the block (counter, 0, particle, axis) under the key (seed, 0)."""
    mask = np.uint64(0xFFFFFFFF)
    c = [np.full(n, counter, np.uint64), np.zeros(n, np.uint64), np.arange(n, dtype=np.uint64),
         np.full(n, axis, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p2 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p2 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p2 & mask,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    u = [(w.astype(np.float64) + 0.5) / 4294967296.0 for w in c[:2]]
    return np.sqrt(-2 * np.log(u[0])) * np.cos(2 * np.pi * u[1])


class _Chain:
    """Nose-Hoover chain of three (Martyna, Tuckerman and Klein 1996), three
    Suzuki-Yoshida weights; half() returns the velocity factor."""

    def __init__(self, kt, tau, dof):
        self.kt, self.dof = kt, dof
        self.q = [dof * kt * tau ** 2, kt * tau ** 2, kt * tau ** 2]
        self.p = [0.0, 0.0, 0.0]

    def _force(self, j, k2):
        return (k2 - self.dof * self.kt if j == 0
                else self.p[j - 1] ** 2 / self.q[j - 1] - self.kt)

    def half(self, ke, dt):
        total = 1.0
        for w in (1.3512071919596577, -1.7024143839193155, 1.3512071919596577):
            h = w * dt / 2
            k2 = 2 * ke
            for sweep in ((2, 1, 0), (0, 1, 2)):
                for j in sweep:
                    s = 1.0 if j == 2 else math.exp(-h / 8 * self.p[j + 1] / self.q[j + 1])
                    self.p[j] = (self.p[j] * s + h / 4 * self._force(j, k2)) * s
                if sweep[0] == 2:
                    f = math.exp(-h / 2 * self.p[0] / self.q[0])
                    k2 *= f * f
            total *= f
            ke *= f * f
        return total


def _trajectory(case, seed):
    s, _, v = _md_inputs(case, seed)
    field = _Field(s)
    con = _Constraints(s) if s.n_constraints else None
    x, v = _t(s.posq[:, :3]), _t(v).T.contiguous()
    m = _t(s.mass)[:, None]
    dt, kt = float(np.float32(2 * FS)), _temperature(case)
    if con:
        v = v + con.velocities(x, v)
    chain = None
    if case["integrator"] == "nvt":
        chain = _Chain(kt, 100 * FS, 3 * s.n - s.n_constraints - 3)
    alpha = math.exp(-dt / U.time(1e-12))
    ke = lambda: float((0.5 * m * v * v).sum())  # noqa: E731
    f = field.all(x)[0]
    for step in range(case["steps"]):
        if chain:
            v = v * chain.half(ke(), dt)
        v = v + f / m * (dt / 2)
        if case["integrator"] == "langevin":
            for part in (0, 1):
                if part:
                    xi = np.stack([_philox_normal(17, step, s.n, c) for c in range(3)], 1)
                    v = alpha * v + torch.sqrt((1 - alpha ** 2) * kt / m) * _t(xi)
                old, x = x, x + v * (dt / 2)
                if con:
                    c = con.positions(x, old)
                    x, v = x + c, v + c / dt
        else:
            old, x = x, x + v * dt
            if con:
                c = con.positions(x, old)
                x, v = x + c, v + c / dt
        if con:
            v = v + con.velocities(x, v)
        scale = chain.half(ke(), dt) if chain else 1.0
        f, _, (pe, _), _ = field.all(x)
        v = (v + f / m * (dt / 2)) * scale
    return dict(x=x, v=v.T.contiguous(), energy=torch.tensor([ke(), float(pe)],
                                                             dtype=torch.float64))


def _splitmix(state):
    state = (state + 0x9E3779B97F4A7C15) & (2 ** 64 - 1)
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & (2 ** 64 - 1)
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & (2 ** 64 - 1)
    return state, z ^ (z >> 31)


def _training(case, seed):
    """Adam on the mean squared error of the 8-64-64-1 tanh network over
    mini-batches in the documented row order, (mul q + add) mod n."""
    x, t, p = (_t(a) for a in _train_inputs(case, seed))
    n = len(x)
    scale = torch.sqrt((x[:, 0] ** 2).mean())
    u = x / scale
    u[:, 5:7] = x[:, 5:7]
    y = (t - x[:, 0]) / scale
    shapes = [(64, 8), (64,), (64, 64), (64,), (64,), (1,)]
    cut = np.cumsum([0] + [int(np.prod(s)) for s in shapes])
    w = p[:-1].clone().requires_grad_(True)

    def net(rows):
        w1, b1, w2, b2, w3, b3 = (w[cut[k]:cut[k + 1]].view(s) for k, s in enumerate(shapes))
        h = torch.tanh(torch.tanh(rows @ w1.T + b1) @ w2.T + b2)
        return h @ w3 + b3[0]

    m1, m2, state, step, losses = torch.zeros_like(w), torch.zeros_like(w), 7, 0, []
    for _ in range(case["epochs"]):
        while True:
            state, z = _splitmix(state)
            mul = (z >> 33) | 1
            if math.gcd(mul, n) == 1:
                break
        state, z = _splitmix(state)
        rows = (torch.arange(n, device=DEV) * mul + z % n) % n
        total = 0.0
        for at in range(0, n, case["batch"]):
            r = rows[at:at + case["batch"]]
            sq = (net(u[r]) - y[r]) ** 2
            total += float(sq.detach().sum())
            (g,) = torch.autograd.grad(sq.mean(), w)
            step += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            lr = 2e-3 * math.sqrt(1 - 0.999 ** step) / (1 - 0.9 ** step)
            with torch.no_grad():
                w -= lr * m1 / (torch.sqrt(m2) + 1e-8)
        losses.append(total / n)
    with torch.no_grad():
        nu = x[:, 0] + scale * net(u)
    return dict(params=torch.cat([w.detach(), scale.view(1)]),
                loss=torch.tensor(losses, dtype=torch.float64), nu=nu)


def exact(case, seed):
    if case["kind"] == "md":
        atoms = case["n"] * {"argon": 1, "water": 3}.get(case["system"], case.get("beads", 1))
        if case["integrator"] == "npt" or case["steps"] * float(atoms) ** 2 > 2.5e10:
            return None
        return _trajectory(case, seed)
    if case["kind"] == "batch":
        return None  # its replicas are the single Langevin cases
    if case["kind"] == "frames":
        rng = np.random.default_rng([seed, case["n"]])
        s, _, posqs = _water(case, rng, case["frames"])
        out = []
        for posq in posqs:
            f, pe, energy, virial = _Field(s).all(_t(posq[:, :3]))
            out.append(dict(f=f, pe=pe, energy=torch.tensor([float(v) for v in energy],
                                                            dtype=torch.float64),
                            virial=torch.tensor([float(v) for v in virial],
                                                dtype=torch.float64)))
        return out
    return _training(case, seed)
