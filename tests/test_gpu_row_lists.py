"""The row lists (a block's j-atoms staged once, a row of indices per
i-atom) at their edges, against the FP64 oracle: one block and less, ragged
last blocks, a box hardly wider than twice the search radius (every atom
has images), the same tilted, a block split into many units and none
(more than 512 blocks); with one interacting type, several with an inert
one, and per-type cutoffs with a switch; with and without Coulomb."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402
from tests.forcecheck import check_forces  # noqa: E402

RC = 8.5e-10
KINDS = ("one", "two and inert", "switched")


def gas(n, n_side, box_m, kind, charged, tilt=0.0, seed=3):
    rng = np.random.default_rng(seed)
    s = systems.argon_lattice(n_atoms=n, n_side=n_side, box_m=box_m, cutoff_m=RC)
    p = s.posq[:, :3].astype(np.float64) + rng.normal(0, 0.3, size=(n, 3))
    s.posq[:, :3] = systems.wrap_into_box(p, s.lattice).astype(np.float32)
    if tilt:
        s = systems.tilted(s, tilt, -tilt, tilt)
    if kind != "one":
        s.types = rng.integers(0, 3, n).astype(np.uint32)
        eps = s.lj.epsilon[0, 0] * np.array([[1.0, 0.7, 0.0], [0.7, 0.5, 0.0], [0.0, 0.0, 0.0]])
        cut = np.full((3, 3), U.length(RC))
        if kind == "switched":
            cut[1, 1] *= 0.8
        rsw = 0.9 * cut if kind == "switched" else cut
        s.lj = systems.LJTable(3, np.full((3, 3), s.lj.sigma[0, 0]), eps, cut, rsw)
    if charged:
        s.posq[:, 3] = np.where(np.arange(n) % 2 == 0, 0.2, -0.2).astype(np.float32)
        rc = U.length(RC)
        s.spme = systems.SpmeParams(systems.ewald_alpha(rc, 1e-5), rc, (64, 64, 64))
    return s


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,n_side,box_m,tilt,charged", [
    (40, 4, 2.3e-9, 0.0, True), (64, 4, 2.3e-9, 0.0, False), (65, 5, 2.3e-9, 0.0, True),
    (216, 6, 2.22e-9, 0.0, False), (343, 7, 2.5e-9, 0.1, True), (4097, 17, 5.8e-9, 0.0, True)])
def test_row_list_edges(oracle, n, n_side, box_m, tilt, charged, kind):
    check(oracle, gas(n, n_side, box_m, kind, charged, tilt), f"{n} atoms, {kind}")


@pytest.mark.parametrize("kind", KINDS)
def test_unsplit_blocks(oracle, kind):
    # 513 blocks, the last with 33 atoms
    check(oracle, gas(512 * 64 + 33, 33, 1.13e-8, kind, False), f"unsplit, {kind}")


def check(oracle, s, tag):
    print("case:", tag, flush=True)
    e = engine_for(s, dt=U.time(2e-15))
    e.force_eval(scalars=True)
    f, sc, got = e.forces(), e.scalars(), e.pairs()
    e.close()

    def keys(p):
        return p[:, 0].astype(np.uint64) << np.uint64(32) | p[:, 1].astype(np.uint64)

    want, band = oracle.pair_set(s.posq, s.lattice, float(s.lj.cutoff.max()) * 1.3)
    missing = np.setdiff1d(keys(want), keys(got))
    if len(band):
        missing = np.setdiff1d(missing, keys(band))
    assert len(missing) == 0
    coul = None if s.spme is None else dict(alpha=s.spme.alpha, r_cut=s.spme.r_cut)
    F, E, W, near = oracle.pair_forces(s.posq, s.types, s.lj.as_dict(), s.lattice, coul=coul,
                                       band=1e-6)
    if s.spme is not None:
        Fr, Er, Wr = oracle.spme_recip(s.posq, s.lattice, s.spme.grid, 4, s.spme.alpha)[:3]
        F, E, W = F + Fr, E + Er, W + Wr
    # the bounds of the FP32 pair terms (1e-5 of a force, see forcecheck);
    # the totals cancel, so they are held to 1e-5 of their terms' sum
    check_forces(f, F, near, tag)
    assert sc["pe"] == pytest.approx(E.sum(), abs=1e-5 * np.abs(E).sum())
    assert sc["virial"] == pytest.approx(W.sum(), abs=1e-5 * np.abs(W).sum())


@pytest.mark.parametrize("n,n_side,box_m", [(40, 4, 2.3e-9), (343, 7, 2.5e-9), (1000, 10, 3.6e-9),
                                            (2197, 13, 4.6e-9), (16400, 26, 9.0e-9)])
@pytest.mark.parametrize("charged", [False, True])
def test_one_type_with_a_switch(oracle, n, n_side, box_m, charged):
    # the general pair terms with a single type: its table and the j types
    # lie behind j-lists of several lengths
    s = gas(n, n_side, box_m, "one", charged)
    cut = np.full((1, 1), U.length(0.95 * RC if charged else RC))
    s.lj = systems.LJTable(1, s.lj.sigma, s.lj.epsilon, cut, 0.85 * cut)
    check(oracle, s, f"{n} atoms, one type, switched")


@pytest.mark.parametrize("pair_list", [0, 1])
def test_neighbor_stats_share_a_unit(pair_list):
    # capacity, largest and total in the same unit: at set-up the capacity is
    # what the largest needed and some headroom
    s = gas(4097, 17, 5.8e-9, "one", False)
    e = engine_for(s, dt=U.time(1e-15), pair_list=pair_list)
    e.force_eval(scalars=False)
    st = e.neighbor_stats()
    e.close()
    print(f"case: list {pair_list}: {st}", flush=True)
    assert 0 < st["max_entries"] <= st["capacity"] <= 4 * st["max_entries"] + 32
    assert st["max_entries"] <= st["entries"]
