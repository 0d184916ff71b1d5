"""Neighbour upkeep at the sizes where its route changes: 1,024 atoms and one
more (the gather inside or behind the one-workgroup binning), 16,384 and one
more (one workgroup or the general path), 1,023 to 1,025 blocks' worth of
units (request cleared by the pair kernel or by its own launch), 512 and 513
blocks (every box tested or a mask).  Each ends in the bits, pair list and
rebuild count of the general path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402
from heddlemd_amd.rng import maxwell_boltzmann  # noqa: E402


@pytest.mark.parametrize("n,side", [(1024, 11), (1025, 11), (8193, 21), (16384, 26), (16385, 26),
                                    (32768, 33), (32769, 33)])
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
    key = lambda p: p[:, 0].astype(np.uint64) << np.uint64(32) | p[:, 1].astype(np.uint64)  # noqa: E731
    assert len(np.setdiff1d(key(want), key(a[4]))) == 0
