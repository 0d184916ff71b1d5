"""The SPME charge spread at its edges against the FP64 oracle: bricks of
every size (grid sides 8 to 96, among them primes' multiples), windows of
more voxels and more atoms than are listed at a time, both spline orders,
and positions that have moved since their voxels were assigned."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402


def ions(n, clustered, grid, order):
    """Point charges without Lennard-Jones terms in a 5 nm box; `clustered`
    of them within about one voxel."""
    rng = np.random.default_rng(n + order)
    rc = U.length(9e-10)
    s = systems.argon_lattice(n_atoms=n, n_side=22, box_m=5.0e-9, cutoff_m=9e-10)
    L = s.lattice[:3]
    p = rng.uniform(-0.5, 0.5, (n, 3)) * L
    p[:clustered] = 0.49 * L + rng.normal(0, 0.8, (clustered, 3))
    s.posq[:, :3] = systems.wrap_into_box(p, s.lattice).astype(np.float32)
    s.posq[:, 3] = np.where(np.arange(n) % 2 == 0, 0.25, -0.25).astype(np.float32)
    s.lj = dataclasses.replace(s.lj, epsilon=np.zeros((1, 1)))
    s.spme = dataclasses.replace(
        systems.SpmeParams(systems.ewald_alpha(rc, 1e-5), rc, grid), order=order)
    return s


def check(oracle, e, s, posq, tag):
    rho, _ = e.spme_grids(s.spme.grid)
    want = oracle.spme_spread(posq, s.lattice, s.spme.grid, s.spme.order)
    err = float(np.abs(rho - want).max() / np.abs(want).max())
    print(f"case: {tag}: grid error {err:.2e}", flush=True)
    # f32 spline weights rounded into 2^-32 fixed point vs the exact sum: a
    # few rounding errors (6e-8) of a cell's largest term
    assert err <= 4e-6


@pytest.mark.parametrize("order", [4, 5])
@pytest.mark.parametrize("grid,n,clustered", [
    ((8, 8, 8), 700, 0), ((32, 32, 32), 4000, 0), ((30, 36, 50), 4000, 0),
    ((48, 40, 96), 4000, 0), ((64, 64, 64), 5000, 0), ((16, 16, 16), 5000, 3500)])
def test_spread_matches_the_oracle(oracle, grid, n, clustered, order):
    s = ions(n, clustered, grid, order)
    e = engine_for(s, dt=U.time(1e-15))
    e.force_eval(scalars=False)
    check(oracle, e, s, s.posq, f"{n} ions, {clustered} clustered, {grid}, order {order}")
    e.close()


@pytest.mark.parametrize("skin_nm", [0.05, 0.3])
def test_spread_of_moved_atoms(oracle, skin_nm):
    s = systems.config_water_8192()
    rng = np.random.default_rng(4)
    v = rng.normal(0, 3e-4, (3, s.n)).astype(np.float32)
    e = engine_for(s, dt=U.time(1e-15), velocities=v, r_skin=U.length(skin_nm * 1e-9))
    for steps in (7, 6):
        e.step(steps)
        check(oracle, e, s, e.positions(), f"moved, skin {skin_nm} nm, {steps} steps")
    e.close()


@pytest.mark.parametrize("axis", range(3))
def test_spread_after_the_box_has_shrunk(oracle, axis):
    # a barostat takes the box to 0.52 of its width; then atoms drift almost
    # half the skin from where they were binned
    s = ions(5000, 0, (40, 40, 40), 4)
    squeeze = dict(pressure=1.0, tau=1.0, compressibility=0.015)
    e = engine_for(s, dt=1.0, velocities=np.zeros((3, s.n), np.float32),
                   berendsen_barostat=squeeze)
    while float(e.lattice()[0]) > 0.52 * float(s.lattice[0]):
        e.step(8)
    e.set_berendsen_barostat(**{**squeeze, "compressibility": 1e-12})
    e.set_positions(e.positions())
    v = np.zeros((3, s.n), np.float32)
    v[axis] = 0.3
    e.set_velocities(v)
    e.step(8)  # 2.4 Bohr, half the skin is 2.55
    width = float(e.lattice()[0]) / float(s.lattice[0])
    s.lattice = np.concatenate([e.lattice()[:3].astype(np.float64), np.zeros(3)])
    check(oracle, e, s, e.positions(), f"box {width:.3f} of its width")
    e.close()
