"""Atoms and results past the pinned transfer size (4 MB), which cross by way of arrays the
context has anyway: the per-atom virial (72 bytes an atom) in several ranges of ids, the
others in one.  Values in id order against the oracle (FP64: forces 1e-11 of their rms,
virial 1e-10 of its rms), positions and velocities bit for bit; and reading them takes no
device memory (the allocator's granularity and the 4 MB of small results aside)."""
import numpy as np
import pytest

from conftest import cu_tables
from test_gpu_parity import CU_MASS, cu_config, frel, make_oracle, make_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(24, 25, 24), (31, 30, 29), (60, 59, 61)])
def test_large_results(oracle_mod, cells):
    import torch
    cfg = cu_config(cells, seed=4)
    order = np.random.Generator(np.random.SFC64(5)).permutation(cfg.n)  # ids in no spatial order
    cfg.r[:], cfg.v[:] = cfg.r[order], cfg.v[order]
    tab = cu_tables(500)
    sim = make_sim(cfg, [CU_MASS])
    sim.eam_alloy_init(tab)
    sim.chunk_neighbors(rcut_max=tab.rc, rcut_inc=0.3)
    sim.zero_force_energy()
    sim.eam_alloy_force(rcut=tab.rc, trigger_thermo_state=True, compute_virial=True)
    sim.force_to_accel()
    sim.ctx.xs_synchronize()
    free = torch.cuda.mem_get_info()[0]
    r, v = sim.state()
    f, vir, ep, rho = sim.forces(), sim.virial(), sim.ep(), sim.rho_dEmb()
    w = np.random.Generator(np.random.SFC64(6)).normal(size=v.shape)
    sim.set_velocities(w)
    assert np.array_equal(sim.state()[1], w)
    sim.set_config(cfg)
    r2, v2 = sim.state()
    assert np.array_equal(r2, cfg.r) and np.array_equal(v2, cfg.v)
    assert free - torch.cuda.mem_get_info()[0] <= 8 << 20
    L = cfg.hi[0] - cfg.lo[0]
    d = r - cfg.r
    assert np.array_equal(v, cfg.v) and np.abs(d - L * np.round(d / L)).max() <= 1e-13 * L.max()
    o = make_oracle(oracle_mod, cfg, [CU_MASS])
    o.set_eam(tab)
    o.build_neighbors(tab.rc, 0.3)
    o.compute_forces("eam")
    ref = o.state()
    assert frel(f, o.forces()) <= 1e-11
    for x, y, tol in ((vir, ref["virial"], 1e-10), (ep, ref["ep"], 1e-10), (rho, ref["rho_dEmb"], 1e-10)):
        assert np.abs(x - y).max() <= tol * np.sqrt((y ** 2).mean())
