"""SPME binning in one workgroup (at most 6,144 atoms and 4,096 bins) and the
reciprocal sums taken by the gather, at the edges of both: a partial round of
atoms per thread, the last size of the path and the first beyond, a full and
an overfull table of bins.  Bars of the other mesh tests (f32 mesh)."""
import numpy as np
import pytest

import oracle
from heddlemd_amd import api, systems
from .gpu_helpers import rel_rms

pytestmark = pytest.mark.gpu

FORCE_TOL, ENERGY_TOL = 1e-5, 1e-6


@pytest.mark.parametrize("n_mol, mesh, brick", [
    (216, (24, 24, 24), (0, 0, 0)), (341, (24, 24, 24), (8, 8, 8)), (342, (32, 24, 20), (4, 4, 4)),
    (1366, (32, 32, 32), (8, 8, 8)), (2048, (48, 48, 48), (0, 0, 0)),
    (2049, (48, 48, 48), (0, 0, 0)), (1024, (64, 64, 64), (4, 4, 4)),
    (1024, (72, 64, 64), (4, 4, 4))])
def test_small_binning(gpu_ctx, n_mol, mesh, brick):
    s = systems.spc_water_n(n_mol, 3 + n_mol)
    ff = systems.water_forcefield(r_cut_nm=0.8, grid=mesh, order=4, exclusions=s["exclusions"])
    if brick[0]:
        ff["spme"]["brick"] = brick
    part = api.ParticleBuffers(gpu_ctx, s["posq"], s["mass"], s["lattice"], types=s["types"])
    field = api.ForceField(gpu_ctx, part, ff)
    posq = s["posq"]
    u_rec, f_rec, _, w_rec = oracle.spme_recip(posq[:, :3], posq[:, 3], s["lattice"], mesh, 4,
                                               ff["coulomb"]["alpha"])
    field.compute(0)                      # force-only: the totals are kept all the same
    u0 = field.spme_scalars()["u_recip"]
    field.compute(1)
    f, sc = field.spme_forces(), field.spme_scalars()
    for h in (field, part):
        h.close()
    errs = rel_rms(f, f_rec), abs(sc["u_recip"] - u_rec) / abs(u_rec)
    print(f"{n_mol} molecules, mesh {mesh}: force {errs[0]:.2e}, U {errs[1]:.2e}")
    assert errs[0] <= FORCE_TOL and errs[1] <= ENERGY_TOL
    assert abs(u0 - u_rec) <= ENERGY_TOL * abs(u_rec)
