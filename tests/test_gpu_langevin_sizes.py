"""The fused Langevin kernels (64 molecules or atoms per workgroup, drawing
waves beside the integrating one) where the last workgroup is full, has one
item or lacks one: the bits, image counts and draw counter of the separate
kernels, eager and through captured step graphs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402


@pytest.mark.parametrize("what,n", [("water", 127), ("water", 128), ("water", 129),
                                    ("water", 89), ("argon", 255), ("argon", 256),
                                    ("argon", 257)])
def test_ragged_last_workgroup(what, n):
    print(f"case: {what} {n}", flush=True)
    if what == "water":
        s = systems.spc_water(n_mol=n, n_side=6, grid=(32, 32, 32), r_cut_m=0.45e-9)
    else:
        s = systems.argon_lattice(n_atoms=n, n_side=7, box_m=2.5e-9, cutoff_m=8.5e-10)
    kt = U.temperature(200.0)
    v0 = np.random.default_rng(n).normal(0, 2e-4, size=(3, s.n)).astype(np.float32)
    out = {}
    for fused in (False, True):
        for graph in (False, True):
            e = engine_for(s, dt=U.time(1e-15), velocities=v0,
                           langevin=dict(friction=1.0 / U.time(1e-13), kt=kt, seed=5))
            e.use_graph(graph)
            e.set_fused_settle(fused)
            e.force_eval(scalars=False)
            e.step(11)
            e.step(3, scalars_last=True)
            p, img = e.positions(images=True)
            out[fused, graph] = (p, img, e.velocities(), e.forces(), e.langevin_counter(),
                                 e.scalars())
            e.close()
    ref = out[False, False]
    assert ref[4] == 14
    for key, o in out.items():
        for k in range(4):
            assert o[k].tobytes() == ref[k].tobytes(), f"{key} output {k}"
        assert o[4:] == ref[4:], key
