"""Two-stage FFT passes for line lengths n1 n2 that are not powers of two:
every register DFT length (2 ... 16) in both stages of the column (a, b) and
row (c) passes, mixed with power-of-two and Stockham axes, against the FP64
oracle on the smallest box of the replica workload."""
import numpy as np
import pytest

import oracle
from .gpu_helpers import rel_rms
from heddlemd_amd import api, systems

pytestmark = pytest.mark.gpu

# f32 rounding of the transform, spread and gather: the bars of the other
# mesh tests (forces 1e-5 relative RMS, energies 1e-6 relative)
FORCE_TOL, ENERGY_TOL = 1e-5, 1e-6


@pytest.mark.parametrize("mesh", [
    (24, 24, 24),      # 4 x 6; c: 12 = 3 x 4
    (18, 20, 24),      # 3 x 6, 4 x 5
    (30, 36, 40),      # 5 x 6, 6 x 6; c: 4 x 5
    (45, 50, 54),      # 5 x 9, 5 x 10; c: 3 x 9
    (60, 72, 80),      # 6 x 10, 8 x 9; c: 5 x 8
    (75, 90, 100),     # 5 x 15, 9 x 10; c: 5 x 10
    (96, 108, 120),    # 8 x 12, 9 x 12; c: 6 x 10
    (144, 150, 48),    # 12 x 12, 10 x 15; c: 4 x 6
    (160, 180, 16),    # 10 x 16, 12 x 15; c: 2 x 4
    (225, 240, 18),    # 15 x 15, 15 x 16; c: 3 x 3
    (162, 25, 20),     # Stockham, 5 x 5; c: 2 x 5
    (64, 48, 250),     # power of two, 6 x 8; c: Stockham (125)
    (24, 32, 8),       # mixed a, power-of-two b; c: 2 x 2
])
def test_mixed_lengths_match_oracle(gpu_ctx, mesh):
    s = systems.spc_water_n(216, 7)
    ff = systems.water_forcefield(r_cut_nm=0.8, grid=mesh, exclusions=s["exclusions"])
    part = api.ParticleBuffers(gpu_ctx, s["posq"], s["mass"], s["lattice"], types=s["types"])
    field = api.ForceField(gpu_ctx, part, ff)
    try:
        u_rec, f_rec, _, w_rec = oracle.spme_recip(s["posq"][:, :3], s["posq"][:, 3],
                                                   s["lattice"], mesh, 4, ff["coulomb"]["alpha"])
        field.compute(1)
        f, sc = field.spme_forces(), field.spme_scalars()
        errs = (rel_rms(f, f_rec), abs(sc["u_recip"] - u_rec) / abs(u_rec),
                abs(sc["w_recip"] - w_rec) / abs(u_rec))
        print(f"mesh {mesh}: force {errs[0]:.2e}, U {errs[1]:.2e}, W/U {errs[2]:.2e}")
        assert errs[0] <= FORCE_TOL and max(errs[1:]) <= ENERGY_TOL
        field.compute(1)   # the same bytes again
        assert np.array_equal(field.spme_forces(), f) and field.spme_scalars() == sc
    finally:
        field.close()
        part.close()
