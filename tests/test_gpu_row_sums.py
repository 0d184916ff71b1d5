"""Rounding of long rows: the f32 sums of the row lists run over at most 64
entries of a lane before they go to fixed point, however long the rows are.

One probe atom feels a near partner's force F and 2,400 atoms on a spherical
cap, each adding just less than half an ulp of F: whatever a lane's f32 sum
takes in behind the partner is lost from it.  The cap's force is what the
forces with and without it differ by."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd import systems, units as U  # noqa: E402
from heddlemd_amd.engine import engine_for  # noqa: E402

NM = U.length(1e-9)
N_CAP, N_INERT = 2400, 16384  # more than 256 blocks: rows are not split
SIGMA, R_NEAR, R_CAP = 0.34 * NM, 0.42 * NM, 0.9 * NM


def lj_force(eps, d):
    """Force on the atom at d from the other."""
    r2 = (d * d).sum(-1, keepdims=True)
    s6 = (SIGMA ** 2 / r2) ** 3
    return 24 * eps * (2 * s6 * s6 - s6) / r2 * d


@pytest.mark.parametrize("axis", range(3))
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_cap_of_small_forces(axis, sign):
    rng = np.random.default_rng(axis + 7)
    L = systems.box_length(9.0 * NM)
    cos = rng.uniform(0.5, 1.0, N_CAP)
    phi = rng.uniform(0, 2 * np.pi, N_CAP)
    cap = np.empty((N_CAP, 3))
    cap[:, axis] = sign * cos
    cap[:, (axis + 1) % 3] = np.sqrt(1 - cos ** 2) * np.cos(phi)
    cap[:, (axis + 2) % 3] = np.sqrt(1 - cos ** 2) * np.sin(phi)
    near = np.zeros((1, 3))
    near[0, axis] = sign * R_NEAR
    # inert atoms out of the others' reach
    inert = rng.uniform(-0.5, 0.5, (2 * N_INERT, 3)) * L
    inert = inert[np.linalg.norm(inert, axis=1) > 2.2 * NM][:N_INERT]
    n = 2 + N_CAP + N_INERT
    posq = np.zeros((n, 4), np.float32)
    posq[:, :3] = systems.wrap_into_box(
        np.concatenate([np.zeros((1, 3)), near, R_CAP * cap, inert]), [L, L, L])
    types = np.repeat(np.arange(4, dtype=np.uint32), [1, 1, N_CAP, N_INERT])
    x = posq[:2 + N_CAP, :3].astype(np.float64)
    big = lj_force(1.0, x[:1] - x[1:2])[0]
    unit = lj_force(1.0, x[:1] - x[2:])
    # each of the cap's forces below 2^-25 F, at least half of it along F
    tiny = np.abs(big[axis]) * 2.0 ** -25 / np.linalg.norm(unit, axis=1).max()
    got = []
    for eps_cap in (tiny, 0.0):
        eps = np.zeros((4, 4))
        eps[0, 1] = eps[1, 0] = 1.0
        eps[0, 2] = eps[2, 0] = eps_cap
        cut = np.full((4, 4), 1.0 * NM)
        s = systems.System(name="cap", posq=posq, mass=np.ones(n, np.float32), types=types,
                           lattice=np.array([L, L, L, 0.0, 0.0, 0.0]),
                           lj=systems.LJTable(4, np.full((4, 4), SIGMA), eps, cut, cut.copy()))
        e = engine_for(s, dt=U.time(1e-15), r_skin=0.1 * NM)
        e.force_eval(scalars=False)
        got.append(e.forces()[0].astype(np.float64))
        e.close()
    want = tiny * unit.sum(0)
    F = np.abs(big[axis])
    lost = np.abs(got[0] - got[1] - want).max() / F
    print(f"case: axis {axis}, sign {sign:+.0f}: cap {np.abs(want).max() / F:.2e} of F, "
          f"lost {lost:.2e} of F", flush=True)
    # 64 entries of at most 2^-25 F each lost in the partner's sum, and the
    # roundings of the two forces to f32 (half an ulp each, 2^-24 F)
    assert lost <= 64 * 2.0 ** -25 + 2 * 2.0 ** -24
