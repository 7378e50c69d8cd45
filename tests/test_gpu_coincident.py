"""Two atoms at the same place: the FP64 forms give what the oracle's square root and
division give there (r = 0, 1/r infinite): the same infinities and NaN, and the other
atoms' values within the usual bounds (1e-11 of rms|F| and of the energies' rms)."""
import dataclasses

import numpy as np
import pytest

from conftest import cu_tables, cuni_tables
from test_gpu_johnson import TA, _oracle_params, _params
from test_gpu_parity import AR_MASS, CU_MASS, lj_params, make_oracle, make_sim

pytestmark = pytest.mark.gpu


def _config(species):
    from exastamp_amd import inputs
    r = np.array([[10.0, 10.0, 10.0], [10.0, 10.0, 10.0], [12.6, 10.0, 10.0], [11.2, 12.3, 10.0],
                  [0.2, 20.0, 20.0], [39.9, 20.0, 22.5], [37.9, 21.0, 21.0]])
    t = (np.arange(len(r)) % species).astype(np.uint8)
    return inputs.Config(r, np.zeros_like(r), t, np.zeros((1, 3)), np.full((1, 3), 40.0))


def _lifted(tab):
    """The tables with r phi(r) other than 0 at r = 0, where phi is then infinite"""
    z = tab.z2r.copy()
    z[:, 0] += 0.3
    return dataclasses.replace(tab, z2r=z)


def _same(x, ref, tol):
    bad = ~np.isfinite(ref)
    assert np.array_equal(x[bad], ref[bad], equal_nan=True) and np.isfinite(x[~bad]).all()
    rms = np.sqrt((ref[~bad] ** 2).mean())
    assert np.abs(x[~bad] - ref[~bad]).max() <= tol * rms


@pytest.mark.parametrize("kind", ["block", "global"])
@pytest.mark.parametrize("pot", ["lj", "johnson", "eam", "eam_lifted", "alloy", "alloy_lifted"])
def test_coincident_atoms(monkeypatch, oracle_mod, pot, kind):
    if kind == "global":
        monkeypatch.setenv("XSMD_LIST", "global")
    else:
        monkeypatch.delenv("XSMD_LIST", raising=False)
    masses = {"lj": [AR_MASS], "johnson": [TA]}.get(pot, [CU_MASS, 58.693] if "alloy" in pot else [CU_MASS])
    cfg = _config(len(masses))
    sim, o = make_sim(cfg, masses), make_oracle(oracle_mod, cfg, masses)
    tab = cuni_tables() if "alloy" in pot else cu_tables(500)
    tab = _lifted(tab) if "lifted" in pot else tab
    rc = {"lj": 8.5, "johnson": 6.1}.get(pot, tab.rc)
    sim.chunk_neighbors(rcut_max=rc, rcut_inc=0.3)
    assert sim.list_info()["kind"] == kind
    o.build_neighbors(rc, 0.3)
    sim.zero_force_energy()
    if pot == "lj":
        eps, sig, _ = lj_params()
        sim.lj_compute_force(parameters={"epsilon": eps, "sigma": sig}, rcut=rc)
        o.set_lj(eps, sig, rc)
        o.compute_forces("lj")
    elif pot == "johnson":
        sim.johnson_force(rcut=rc, parameters=_params(), compute_virial=True)
        o.set_johnson(_oracle_params(), rc)
        o.compute_forces("johnson")
    else:
        sim.eam_alloy_init(tab)
        sim.eam_alloy_force(rcut=rc, trigger_thermo_state=True, compute_virial=True)
        o.set_eam(tab)
        o.compute_forces("eam")
    sim.force_to_accel()
    ref = o.state()
    assert not np.isfinite(ref["ep"][:2]).any() and np.isfinite(ref["ep"][2:]).all()
    _same(sim.ep(), ref["ep"], 1e-11)
    _same(sim.forces(), o.forces(), 1e-11)
    _same(sim.virial().reshape(-1), ref["virial"].reshape(-1), 1e-10)
