"""SPME binning in one workgroup (at most 5,120 atoms and 4,096 bins) and the
reciprocal sums taken by the gather, at the edges of both: a partial round of
atoms per thread, the last size of the path and the first beyond, a full and
an overfull table of bins.  Bars of the other mesh tests (f32 mesh)."""
import numpy as np
import pytest

import oracle
from heddlemd_amd import api, systems
from .gpu_helpers import oracle_pair, rel_rms

pytestmark = pytest.mark.gpu

FORCE_TOL, ENERGY_TOL = 1e-5, 1e-6


@pytest.mark.parametrize("n_mol, mesh, brick", [
    (216, (24, 24, 24), (0, 0, 0)), (341, (24, 24, 24), (8, 8, 8)), (342, (32, 24, 20), (4, 4, 4)),
    (1366, (32, 32, 32), (8, 8, 8)), (1706, (48, 48, 48), (0, 0, 0)),
    (1707, (48, 48, 48), (0, 0, 0)), (2048, (48, 48, 48), (0, 0, 0)),
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
    errs = (rel_rms(f, f_rec), abs(sc["u_recip"] - u_rec) / abs(u_rec),
            abs(sc["w_recip"] - w_rec) / abs(u_rec))
    print(f"{n_mol} molecules, mesh {mesh}: force {errs[0]:.2e}, U {errs[1]:.2e}, "
          f"W/U {errs[2]:.2e}")
    assert errs[0] <= FORCE_TOL and max(errs[1:]) <= ENERGY_TOL
    assert abs(u0 - u_rec) <= ENERGY_TOL * abs(u_rec)


@pytest.mark.parametrize("mesh, bricks", [
    ((48, 48, 48), [(8, 8, 8), (24, 12, 12)]),    # 336 partials x 216 and 32 bricks
    ((72, 72, 72), [(8, 8, 8), (4, 4, 4)]),       # 360 x 729 and 360 x 5,832: the sum's launch
    ((64, 48, 250), [(8, 8, 10), (4, 4, 5)])])    # the power-of-two a axis, both ways
def test_reciprocal_sums_in_the_gather_or_before(gpu_ctx, mesh, bricks):
    """The reciprocal virial that every workgroup of the gather hands out per
    atom, summed by the workgroup or (partials times bricks above 3 * 2^19) by
    a launch before: the same bytes, and the oracle's total.  Bar of the total:
    f32 terms of the pair virial and W / n rounded once per atom."""
    s = systems.spc_water_n(216, 5)
    posq = s["posq"]
    out = []
    for brick in bricks:
        ff = systems.water_forcefield(r_cut_nm=0.8, grid=mesh, order=4,
                                      exclusions=s["exclusions"])
        ff["spme"]["brick"] = brick
        part = api.ParticleBuffers(gpu_ctx, posq, s["mass"], s["lattice"], types=s["types"])
        field = api.ForceField(gpu_ctx, part, ff)
        field.compute(1)
        e, w = (x.copy() for x in part.energies())
        out.append((field.spme_scalars(), e, w, part.forces().copy()))
        for h in (field, part):
            h.close()
    u_rec, _, _, w_rec = oracle.spme_recip(posq[:, :3], posq[:, 3], s["lattice"], mesh, 4,
                                           ff["coulomb"]["alpha"])
    _, _, w_pair = oracle_pair(s, ff, posq)
    for sc, e, w, f in out:
        total = float(w.astype(np.float64).sum())
        want = float(w_pair.sum()) + w_rec
        print(f"mesh {mesh}: W {abs(sc['w_recip'] - w_rec) / abs(u_rec):.2e}, "
              f"total {abs(total - want) / abs(want):.2e}")
        assert abs(sc["w_recip"] - w_rec) <= ENERGY_TOL * abs(u_rec)
        assert abs(total - want) <= 5e-6 * (np.abs(w_pair).sum() + abs(w_rec))
        assert sc == out[0][0]
        for a, b in ((e, out[0][1]), (w, out[0][2]), (f, out[0][3])):
            assert a.tobytes() == b.tobytes()
