"""Neighbour upkeep at the sizes where its route changes: 1,024 atoms and one
more (the gather inside or behind the one-workgroup binning) and 16,384 (its
largest) against the general path, in bits, pair list and rebuild count;
16,385 atoms, 512 and 513 blocks (every box tested or a mask), 1,024 and 1,025
units (request cleared by the pair kernel, or by its own launch that also
orders the units) eager against captured, in bits, and against the FP64
oracle after several rebuilds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402
from heddlemd_amd.rng import maxwell_boltzmann  # noqa: E402
from tests.forcecheck import check_forces  # noqa: E402


def key(p):
    return p[:, 0].astype(np.uint64) << np.uint64(32) | p[:, 1].astype(np.uint64)


@pytest.mark.parametrize("n,side", [(16385, 26), (32768, 33), (32769, 33), (65536, 41),
                                    (65537, 41)])
def test_general_path(oracle, n, side):
    s = systems.argon_lattice(n_atoms=n, n_side=side, box_m=side * 3.45e-10)
    v = maxwell_boltzmann(s.mass, U.temperature(250.0), seed=2)
    out = []
    for graph in (False, True):
        e = engine_for(s, dt=U.time(4e-15), velocities=v)
        e.use_graph(graph)
        e.step(70)
        e.step(10, scalars_last=True)
        out.append((e.positions(), e.velocities(), e.forces(), e.scalars(), e.pairs()))
        e.close()
    a, b = out
    print(f"case: {n} atoms, rebuilds {a[3]['rebuilds']:.0f}", flush=True)
    assert a[3]["rebuilds"] >= 4  # two of them at set-up
    for k in range(3):
        assert a[k].tobytes() == b[k].tobytes()
    assert a[3] == b[3]
    assert np.array_equal(a[4], b[4])
    want, band = oracle.pair_set(a[0], s.lattice, float(s.lj.cutoff.max()))
    missing = np.setdiff1d(key(want), key(a[4]))
    if len(band):
        missing = np.setdiff1d(missing, key(band))
    assert len(missing) == 0
    F, _, _, near = oracle.pair_forces(a[0], s.types, s.lj.as_dict(), s.lattice, band=1e-6)
    check_forces(a[2], F, near, f"{n} atoms")


@pytest.mark.parametrize("n,side", [(1024, 11), (1025, 11), (8193, 21), (16384, 26)])
@pytest.mark.parametrize("langevin", [False, True])
def test_routes_agree(oracle, n, side, langevin):
    s = systems.argon_lattice(n_atoms=n, n_side=side, box_m=side * 3.45e-10)
    kt = U.temperature(250.0)
    out = []
    for small in (True, False):
        kw = dict(langevin=dict(friction=1.0 / U.time(1e-13), kt=kt, seed=3)) if langevin else {}
        e = engine_for(s, dt=U.time(4e-15), velocities=maxwell_boltzmann(s.mass, kt, seed=2), **kw)
        e.set_small_neighbor(small)
        e.step(70)
        e.step(10, scalars_last=True)
        out.append((e.positions(), e.velocities(), e.forces(), e.scalars(), e.pairs()))
        e.close()
    a, b = out
    print(f"case: {n} atoms, rebuilds {a[3]['rebuilds']:.0f}", flush=True)
    assert a[3]["rebuilds"] >= 2
    for k in range(3):
        assert a[k].tobytes() == b[k].tobytes()
    assert a[3] == b[3]
    assert np.array_equal(a[4], b[4])
    # the list of the last rebuild still holds every pair within the cutoff
    want, band = oracle.pair_set(a[0], s.lattice, float(s.lj.cutoff.max()))
    assert len(np.setdiff1d(key(want), key(a[4]))) == 0
