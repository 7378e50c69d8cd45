"""Newton-symmetric operators: the two atoms of a pair get opposite forces.

Three thousand boxes of two atoms each.  Inside a box both atoms see the same distance,
and the pair scalar is symmetric in them: their forces are opposite to the last bit, in
both precisions, for one species and for two.  Through a periodic image the displacement
rounds differently from either atom, by at most an ulp of the box's edge (2e-15 of r);
with pair forces no steeper than d ln F / d ln r of 100 that is 1e-12 of the largest force
in FP64, and an ulp of the rounded knot fraction, 1e-6, in the mixed form."""
import numpy as np
import pytest

from conftest import cu_tables, cuni_tables
from test_gpu_parity import AR_MASS, CU_MASS, lj_params, make_sim

pytestmark = pytest.mark.gpu

REPS, EDGE = 3000, 16.0


def _pairs(species, image, rmax, seed=7):
    from exastamp_amd import inputs
    g = inputs.rng(seed)
    u = g.normal(size=(REPS, 3))
    u /= np.sqrt((u * u).sum(1))[:, None]
    a = g.uniform(5.0, 11.0, size=(REPS, 3))
    if image:  # the second atom beyond an x face
        a[:, 0] = np.where(u[:, 0] < 0, 0.1, EDGE - 0.1) + g.uniform(-0.05, 0.05, size=REPS)
        u[:, 0] = np.sign(u[:, 0]) * np.maximum(np.abs(u[:, 0]), 0.5)
    b = a + u * g.uniform(2.0, rmax, size=REPS)[:, None]
    b[:, 0] -= EDGE * np.floor(b[:, 0] / EDGE)
    assert (np.abs(b - a).max(1) > 0.5 * EDGE).all() == image
    r = np.stack([a, b], 1).reshape(-1, 3)
    t = g.integers(0, species, size=2 * REPS).astype(np.uint8)
    hi = np.full((REPS, 3), EDGE)
    return inputs.Config(r, np.zeros_like(r), t, np.zeros((REPS, 3)), hi, (1, 1, 1),
                         np.repeat(np.arange(REPS, dtype=np.uint16), 2))


@pytest.mark.parametrize("kind", ["block", "global"])
@pytest.mark.parametrize("image", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("pot", ["lj", "cu", "cuni"])
def test_pair_forces_are_opposite(monkeypatch, pot, mixed, image, kind):
    if kind == "global":
        monkeypatch.setenv("XSMD_LIST", "global")
    else:
        monkeypatch.delenv("XSMD_LIST", raising=False)
    masses = {"lj": [AR_MASS], "cu": [CU_MASS], "cuni": [CU_MASS, 58.693]}[pot]
    cfg = _pairs(len(masses), image, 4.0)
    sim = make_sim(cfg, masses)
    sim.chunk_neighbors(rcut_max=4.95, rcut_inc=0.3)
    assert sim.list_info()["kind"] == kind
    sim.zero_force_energy()
    if pot == "lj":
        eps, _, _ = lj_params()
        sim.lj_compute_force_symetric(parameters={"epsilon": eps, "sigma": 2.3}, rcut=4.95, mixed=mixed)
    else:
        tab = cu_tables() if pot == "cu" else cuni_tables()
        sim.eam_alloy_init(tab)
        sim.eam_alloy_force(rcut=tab.rc, trigger_thermo_state=True, mixed=mixed, eam_symmetry=True)
    f = sim.accelerations().reshape(REPS, 2, 3)  # forces: force_to_accel has not run
    assert np.abs(f).max(axis=(1, 2)).min() > 0.0
    net = np.abs(f.sum(1)).max()
    assert net <= ((1e-6 if mixed else 1e-12) * np.abs(f).max() if image else 0.0)
