"""Capacities of the row lists: headroom for frames and steps that get
denser, unsplit blocks (more than 256) and split ones, lists that grow from
nothing, and no more memory than what is needed when long cutoffs split the
blocks."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402


def keys(p):
    return p[:, 0].astype(np.uint64) << np.uint64(32) | p[:, 1].astype(np.uint64)


def free_bytes():
    """Of the HIP runtime that libheddle links."""
    hip = C.CDLL("/opt/rocm/lib/libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def complete(oracle, e, posq, lattice, cutoff):
    want, band = oracle.pair_set(posq, lattice, cutoff)
    missing = np.setdiff1d(keys(want), keys(e.pairs()))
    if len(band):
        missing = np.setdiff1d(missing, keys(band))
    return len(missing) == 0


@pytest.mark.parametrize("n,side", [(4000, 16), (17000, 26)])
def test_imploding_gas(oracle, n, side):
    # the gas of the contract test, in split blocks and in unsplit ones: the
    # list grows between graph launches and holds every pair at the end
    print(f"case: {n} imploding", flush=True)
    s = systems.argon_lattice(n_atoms=n, n_side=side, box_m=(side + 1) * 3.4e-10)
    s.lj.epsilon[:] = 0.0
    dt = U.time(1e-15)
    x0 = s.posq[:, :3].astype(np.float64)
    v = (-0.45 * x0 / (400 * dt)).T.astype(np.float32)
    e = engine_for(s, dt=dt, velocities=v)
    e.force_eval(scalars=False)
    e.step(400)
    p = e.positions()
    assert np.abs(p[:, :3] - (x0 + 400 * dt * v.T.astype(np.float64))).max() < 1e-3
    assert complete(oracle, e, p, s.lattice, 0.4 * float(s.lj.cutoff.max()))
    e.close()


@pytest.mark.parametrize("step", [False, True])
@pytest.mark.parametrize("n_mol,side,skin_nm", [(2646, 14, 0.27), (8192, 21, 0.27),
                                                (8192, 21, 0.2), (8192, 21, 0.24)])
def test_denser_frame(oracle, n_mol, side, skin_nm, step):
    # a frame 1.4 times as dense behind the set-up's, in one context; at a
    # skin of 0.24 nm the LDS leaves an unsplit block less headroom than that
    print(f"case: {n_mol} molecules, skin {skin_nm} nm, 1.4 times as dense", flush=True)
    s = systems.spc_water(n_mol=n_mol, n_side=side, grid=(40, 40, 40))
    s.water_groups = None
    e = engine_for(s, dt=U.time(1e-20), r_skin=skin_nm * 1e-9 * U.length(1.0))
    e.force_eval(scalars=False)
    p = s.posq.copy()
    p[:, :3] = systems.wrap_into_box(p[:, :3].astype(np.float64) * 1.4 ** (-1 / 3), s.lattice)
    e.set_positions(p)
    if step:
        e.step(1)
    else:
        e.force_eval(scalars=False)
    assert complete(oracle, e, p, s.lattice, float(s.lj.cutoff.max()))
    e.close()


def test_pairs_from_none(oracle):
    # 192 atoms far apart at set-up, one cluster in the next frame
    print("case: 192 atoms, apart and clustered", flush=True)
    s = systems.argon_lattice(n_atoms=192, n_side=6, spacing_m=3.0e-9, box_m=1.8e-8)
    e = engine_for(s, dt=U.time(1e-15))
    e.force_eval(scalars=False)
    p = s.posq.copy()
    p[:, :3] *= np.float32(0.12)
    e.set_positions(p)
    e.force_eval(scalars=False)
    assert complete(oracle, e, p, s.lattice, float(s.lj.cutoff.max()))
    e.close()


def test_memory_of_a_long_cutoff():
    # 1.2 nm splits the blocks of 24,576 atoms; the rows hold about 1,600
    # neighbours of 2 bytes, half as many again, 128 and the padding of each
    # part
    s = systems.spc_water(n_mol=8192, n_side=21, grid=(64, 64, 64), r_cut_m=1.2e-9)
    engine_for(s, dt=U.time(1e-15)).close()
    before = free_bytes()
    e = engine_for(s, dt=U.time(1e-15))
    used = before - free_bytes()
    st = e.neighbor_stats()
    e.close()
    print(f"case: 24,576 atoms, r_cut 1.2 nm: {used / 2 ** 20:.0f} MiB, {st}", flush=True)
    assert used <= 300 * 2 ** 20


def test_split_blocks_are_joined_again():
    # a frame that splits the blocks, then the set-up's again: the lists end
    # as those of a context that never saw the dense frame, bits included
    print("case: 8192 molecules, dense frame and back", flush=True)
    s = systems.spc_water(n_mol=8192, n_side=21, grid=(40, 40, 40))
    s.water_groups = None
    dense = s.posq.copy()
    dense[:, :3] = systems.wrap_into_box(dense[:, :3].astype(np.float64) * 1.4 ** (-1 / 3),
                                         s.lattice)
    moved = s.posq.copy()  # far enough for a rebuild
    moved[:, :3] = systems.wrap_into_box(moved[:, :3].astype(np.float64) + 4.0, s.lattice)
    out = []
    for frames in ([s.posq], [dense, s.posq, moved, s.posq, moved, s.posq]):
        e = engine_for(s, dt=U.time(1e-15), r_skin=0.2e-9 * U.length(1.0))
        units = []
        for p in frames:
            e.set_positions(p)
            e.force_eval(scalars=True)
            units.append(e.neighbor_stats()["max_entries"])
        st, sc = e.neighbor_stats(), e.scalars()
        out.append((st["max_entries"], st["entries"], e.forces().tobytes(), sc["pe"]))
        e.close()
        print(f"  most of a unit, frame by frame: {units}", flush=True)
    assert units[1] < 0.75 * units[-1]  # still split behind the dense frame
    assert out[0] == out[1]
