"""The bunch kernels' deposits: boxes shaped by what a block covers, one, four
and sixteen particles per lane, partly filled last blocks."""
import numpy as np
import pytest

from helpers import normwise

pytestmark = pytest.mark.gpu

CR, CZ, D = 96, 64, 5e-4


def _bunch(rows, n, seed=9):
    rng = np.random.default_rng(seed)
    r = D * (0.6 + (rows - 1.2) * np.sqrt(rng.random(n)))
    z = np.sort(D * (2 + 40 * rng.random(n)))  # in the order of injection
    v = rng.standard_normal((2, n)) * 1e6
    return r, z, v[0], v[1], np.full(n, 2.7e8), rng.uniform(0.5, 1.5, n) * 1e3


def _sim(precision, arrs):
    from pdp3_amd import capi

    sim = capi.Simulation(CR + 1, CZ + 1, CR * D, CZ * D, 0.5 * D / 3e8, precision=precision)
    sim.boundary_conditions()
    sim.set_field("E_r", 1e4 * np.random.default_rng(1).standard_normal((CR + 1, CZ + 1)))
    sim.add_bunch_loaded(-1, 1.0, *arrs)
    return sim


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("rows,n", [
    (2, 3001),
    (13, 3001), (14, 3001),  # 16 x 32 nodes hold 13 rows of cells
    (29, 3001), (30, 3001),  # 32 x 16
    (61, 3001), (62, 3001),  # 64 x 8
    (90, 3001),              # more than any shape
    (20, 1 << 20), (20, (1 << 20) + 77),  # four per lane
    (20, (1 << 22) + 1029),               # sixteen
])
def test_step_of_a_bunch_in_any_order(precision, rows, n):
    """A bunch in the order of injection, whose blocks cover few columns and so
    take the box that holds their rows, against the same particles in random
    order, whose blocks cover all of it, and in the FP64 form against the split
    entry points too: the same arithmetic per particle, so J and rho differ by
    the order of their FP64 sums only (some 2e3 terms of either sign a node at
    most, 2e3 x 1e-16 x sqrt(2e3) of the largest sum: 1e-10 holds)."""
    arrs = _bunch(rows, n)
    p = np.random.default_rng(2).permutation(n)
    names = ("J_r", "J_phi", "J_z", "rho_bunch")
    out = []
    for a in (arrs, tuple(x[p] for x in arrs)):
        sim = _sim(precision, a)
        sim.step(1)
        out.append({k: sim.field(k) for k in names})
        sim.close()
    if precision == 0:
        sim = _sim(precision, arrs)
        sim.h_calc()
        sim.reset_j()
        sim.step_v(0)
        sim.full_current_distribution(0)
        sim.charge_weighting(0)
        out.append({k: sim.field(k) for k in names})
        sim.close()
    for other in out[1:]:
        for k in names:
            assert normwise(out[0][k], other[k]) <= 1e-10, (k, normwise(out[0][k], other[k]))
