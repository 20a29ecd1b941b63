"""SPME spread and gather at the edges of the brick scheme: one, two and more
bricks an axis, each spline order, bricks with more atoms than the spread's
queue holds, an uncharged atom, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from heddlemd_amd import api, systems
from .gpu_helpers import rel_rms

pytestmark = pytest.mark.gpu

# f32 spread, transform and gather (the bars of the other mesh tests)
FORCE_TOL, ENERGY_TOL = 1e-5, 1e-6


@pytest.mark.parametrize("order,mesh,brick", [
    (4, (8, 8, 8), (8, 8, 8)),          # a single brick: 648 atoms through one queue
    (4, (8, 16, 24), (8, 8, 8)),        # one, two and three bricks
    (4, (20, 16, 12), (4, 4, 4)),       # bricks as narrow as the support
    (4, (32, 32, 32), (16, 16, 8)),
    (5, (10, 20, 30), (10, 10, 6)),
    (6, (12, 24, 36), (12, 6, 6)),
    (6, (40, 40, 40), (8, 8, 8)),
    (8, (16, 16, 32), (16, 8, 8)),
])
def test_spread_and_gather_match_oracle(gpu_ctx, order, mesh, brick):
    s = systems.spc_water_n(216, 11)
    posq = s["posq"].copy()
    posq[5, 3] = 0.0
    ff = systems.water_forcefield(r_cut_nm=0.8, grid=mesh, order=order,
                                  exclusions=s["exclusions"])
    ff["spme"]["brick"] = brick
    part = api.ParticleBuffers(gpu_ctx, posq, s["mass"], s["lattice"], types=s["types"])
    field = api.ForceField(gpu_ctx, part, ff)
    try:
        u_rec, f_rec, _, _ = oracle.spme_recip(posq[:, :3], posq[:, 3], s["lattice"], mesh,
                                               order, ff["coulomb"]["alpha"])
        field.compute(1)
        err_f = rel_rms(field.spme_forces(), f_rec)
        err_u = abs(field.spme_scalars()["u_recip"] - u_rec) / abs(u_rec)
        rho, _ = field.spme_grids(mesh)
        q = float(posq[:, 3].astype(np.float64).sum())
        print(f"order {order} mesh {mesh} brick {brick}: force {err_f:.2e}, U {err_u:.2e}")
        assert err_f <= FORCE_TOL and err_u <= ENERGY_TOL
        # every atom's charge once: f32 weights and one rounding a mesh point
        assert abs(float(rho.astype(np.float64).sum()) - q) <= 1e-5 * np.abs(posq[:, 3]).sum()
        field.compute(1)   # the same mesh whatever order the bins were filled in
        assert np.array_equal(field.spme_grids(mesh)[0], rho)
    finally:
        field.close()
        part.close()
