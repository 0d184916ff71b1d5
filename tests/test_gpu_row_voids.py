"""Row lists beside a void: a few vapour atoms share a block with each other
and with the liquid's surface, so their boxes span much of the liquid.  The
lists must hold the atoms near the block's atoms, not those near its box:
frames with vapour follow a frame without in the same context, and the forces
are the FP64 oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402
from tests.forcecheck import check_forces  # noqa: E402

NM = U.length(1e-9)
A = 0.37 * NM  # lattice spacing of the liquid


def sites(shape, side, n, rng):
    """n lattice sites (in units of A) of a slab or a droplet of edge `side`,
    each displaced by a few percent."""
    m = 2 * side
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) - (m - 1) / 2
    if shape == "slab":
        g = g[(np.abs(g[:, :2]) < side / 2).all(axis=1)]
        order = np.argsort(np.abs(g[:, 2]), kind="stable")
    else:
        order = np.argsort((g * g).sum(1), kind="stable")
    return g[order][:n] + rng.uniform(-0.04, 0.04, (n, 3))


@pytest.mark.parametrize("shape,side,n", [("slab", 20, 7959), ("slab", 27, 19000),
                                          ("droplet", 22, 9001), ("droplet", 30, 21000)])
def test_vapour_beside_liquid(oracle, shape, side, n):
    rng = np.random.default_rng(n)
    x = A * sites(shape, side, n, rng)
    L = np.array([side * A, side * A, 3 * side * A] if shape == "slab" else 3 * [2.2 * side * A])
    L = np.array([systems.box_length(v) for v in L])
    s = systems.argon_lattice(n_atoms=n, n_side=40, cutoff_m=8.5e-10)
    s.lattice = np.concatenate([L, np.zeros(3)])
    s.posq[:, :3] = systems.wrap_into_box(x, L)
    e = engine_for(s, dt=U.time(1e-15))
    for vapour in (0, 9, 30, 17):
        p = s.posq.copy()
        free = []
        while len(free) < vapour:
            y = rng.uniform(-0.5, 0.5, 3) * L
            d = np.concatenate([x[:n - vapour], np.array(free).reshape(-1, 3)]) - y
            d -= L * np.rint(d / L)
            if (d * d).sum(1).min() > (1.2 * A) ** 2:
                free.append(y)
        if vapour:
            p[n - vapour:, :3] = systems.wrap_into_box(np.array(free), L)
            e.set_positions(p)
        print(f"case: {shape}, {n} atoms, {vapour} in the vapour", flush=True)
        e.force_eval(scalars=True)
        F, E, W, near = oracle.pair_forces(p, s.types, s.lj.as_dict(), s.lattice, band=1e-6)
        check_forces(e.forces(), F, near, f"{shape} {vapour}")
        assert e.scalars()["pe"] == pytest.approx(E.sum(), abs=1e-5 * np.abs(E).sum())
    e.close()


def test_block_that_meets_most_blocks_in_several_images():
    # a dense cluster in a box hardly wider than twice the search radius, and
    # 40 atoms around it: their blocks meet 512 others in about 1,500 images
    rng = np.random.default_rng(2)
    m, a, side = 32, 0.2 * NM, 12.0 * NM
    L = np.full(3, systems.box_length(side))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) - (m - 1) / 2
    f = rng.uniform(-0.5, 0.5, (800, 3)) * L
    f = f[np.abs(f).max(axis=1) > (m / 2 + 1.5) * a][:40]
    x = np.concatenate([a * (g + rng.uniform(-0.04, 0.04, g.shape)), f])
    n = len(x)
    s = systems.argon_lattice(n_atoms=n, n_side=40, sigma_m=0.18e-9, cutoff_m=5.7e-9)
    s.lattice = np.concatenate([L, np.zeros(3)])
    s.posq[:, :3] = systems.wrap_into_box(x, L)
    out = []
    for pair_list in (0, 1):
        print(f"case: {n} atoms, list {pair_list}", flush=True)
        e = engine_for(s, dt=U.time(1e-15), r_skin=0.2 * NM, pair_list=pair_list)
        e.force_eval(scalars=True)
        out.append((e.forces().astype(np.float64), e.count_pairs(), e.scalars()["pe"]))
        e.close()
    (fr, nr, er), (fa, na, ea) = out
    # pairs within rounding of the cutoff may fall on either side
    assert abs(int(nr) - int(na)) <= 1e-6 * na
    check_forces(fr, fa, None, "rows and atom lists")
    assert er == pytest.approx(ea, rel=1e-5)
