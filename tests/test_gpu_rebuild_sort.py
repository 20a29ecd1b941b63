"""The list rebuild's cell sort at the sizes where its paths change: one
workgroup up to 12,288 atoms (2^3 .. 32^3 cells, several atoms a thread, a
partial last round), four launches beyond; and clustered atoms, whose cells
hold many.  The pair set is exact; the cells fill in arbitrary order, and the
rank that puts the atoms of each into the order of their ids shows in the bits
of the forces, equal from build to build."""
import numpy as np
import pytest

import oracle
from heddlemd_amd import api, systems
from heddlemd_amd import units as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, clustered", [
    (1, False), (2, False), (64, False), (65, True), (520, False), (1025, True), (4097, False),
    (5120, False), (5121, True), (6553, False), (6554, False), (12288, True), (12289, False), (20001, True)])
def test_pair_set_and_order(gpu_ctx, n, clustered):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    s = systems.argon(n, side, max(3.0, 7.84 / 22 * side))
    L = float(s["L"])
    pos = s["posq"][:, :3].astype(np.float64) + rng.uniform(-0.05, 0.05, (n, 3)) * U.NM
    if clustered:                            # empty cells, and several atoms in the others
        pos *= 0.7
    pos = (pos + rng.uniform(0, 1, 3) * L + 0.5 * L) % L - 0.5 * L
    posq = np.concatenate([pos, np.zeros((n, 1))], 1).astype(np.float32)
    part = api.ParticleBuffers(gpu_ctx, posq, s["mass"], s["lattice"], types=s["types"])
    field = api.ForceField(gpu_ctx, part, s["ff"])
    field.compute(0)
    f0 = part.forces().copy()
    got = field.pair_snapshot()
    rs = np.float32(s["ff"]["lj"]["cutoff"][0]) + np.float32(s["ff"]["r_skin"])
    want = oracle.pair_set_f32(posq, s["lattice"].astype(np.float32), rs * rs, cells=n > 4000)
    same = []
    for _ in range(3):                       # the same list built again
        gen = field.stats()["generation"]
        field.request_rebuild()
        field.compute(0)
        assert field.stats()["generation"] == gen + 1
        same.append(part.forces().tobytes() == f0.tobytes())
    for h in (field, part):
        h.close()
    assert got.shape == want.shape and np.array_equal(got, want)
    assert all(same)
