"""The pair kernel's two ways to share a list, either side of the number of
entries where they change (1,536): a workgroup per entry for shorter lists,
whole entries per wave for longer ones.  Forces and energies against the FP64
oracle, and the same bytes for every launch shape: 256 and 512 workgroups, which
take several entries and clusters each, and as many as the list has work for.

Force tolerance: both atoms of a pair are moved to the image nearest a cluster
centre in f32, each by up to an ulp of L/2; at the lattice spacing a the r^-13
of LJ turns that into 2 x 13 ulp(L/2) / a of the pair force (1.5e-5 at 1,000
atoms, where 8.1e-6 is measured).  Energies: 5e-6 (f32 terms, no steep
cancellation)."""
import numpy as np
import pytest

from heddlemd_amd import api, systems
from tests.gpu_helpers import oracle_pair, rel_rms

pytestmark = pytest.mark.gpu


def jittered_argon(n, charged):
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    s = systems.argon(n, side, max(2.6, 7.84 / 22 * side))
    rng = np.random.default_rng(n)
    L = float(s["L"])
    pos = s["posq"][:, :3] + rng.normal(scale=0.01 * L / side, size=(n, 3)) + rng.uniform(0, L, 3)
    pos = (pos + 0.5 * L) % L - 0.5 * L
    q = 0.05 * (1.0 - 2.0 * (np.arange(n) % 2)) * charged
    s["posq"] = np.concatenate([pos, q[:, None]], 1).astype(np.float32)
    if charged:
        rc = s["ff"]["lj"]["cutoff"][0]
        s["ff"] = dict(s["ff"], coulomb={"alpha": 3.0 / rc, "r_cut": rc, "k_coulomb": 1.0})
    off = np.zeros(n + 1, np.uint32)         # every third atom excludes its successor
    par = []
    for i in range(n):
        off[i] = len(par)
        if i % 3 == 0 and i + 1 < n:
            par.append(i + 1)
        elif i % 3 == 1:
            par.append(i - 1)
    off[n] = len(par)
    s["ff"] = dict(s["ff"], exclusions=(off, np.asarray(par, np.uint32)))
    return s, 26.0 * float(np.spacing(np.float32(0.5 * L))) / (L / side)


@pytest.mark.parametrize("n, charged, shared", [
    (1, 0, True), (63, 1, True), (130, 0, True), (1000, 1, True), (8000, 0, True),
    (8000, 1, True), (12500, 0, True), (12500, 1, True), (17000, 1, False)])
def test_forces_and_launch_shapes(gpu_ctx, n, charged, shared):
    s, tol = jittered_argon(n, charged)
    part = api.ParticleBuffers(gpu_ctx, s["posq"], s["mass"], s["lattice"], types=s["types"])
    field = api.ForceField(gpu_ctx, part, s["ff"])
    field.compute(1)
    f, (e, _) = part.forces().copy(), part.energies()
    entries = field.stats()["n_work"]
    base = field.tuning()
    same = []
    for blocks in (1, 2, 32):
        field.set_tuning(dict(base, pair_blocks_per_cu=blocks))
        field.compute(1)
        same.append(part.forces().tobytes() == f.tobytes())
    field.compute(0)
    err_f0 = rel_rms(part.forces(), f) if n > 1 else 0.0
    for h in (field, part):
        h.close()
    f_ref, e_ref, _ = oracle_pair(s, s["ff"], s["posq"])
    err = rel_rms(f, f_ref) if n > 1 else float(np.abs(f).max())
    err_e = abs(e.astype(np.float64).sum() - e_ref.sum()) / max(np.abs(e_ref).sum(), 1e-30)
    print(f"{n} atoms, {entries} entries: forces {err:.2e}, energy {err_e:.2e}, "
          f"without energies {err_f0:.2e}")
    assert (entries < 1536) == shared
    if n >= 8000:
        assert entries > 2 * 256          # several entries a workgroup of both small grids
    assert all(same)
    assert err <= tol and err_e <= 5e-6 and err_f0 <= 1e-6
