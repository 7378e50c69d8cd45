"""Pieces of the FP64 passes and of the list build where they meet: distances and
reciprocals one by one, lanes whose neighbour has no atom or a much longer list, the cell
sort on both sides of its one-kernel form, the smallest spline tables of the adjoint."""
import numpy as np
import pytest

import test_gpu_adjoint_sweeps as sweeps
from conftest import cu_tables, cuni_tables
from test_gpu_parity import CU_MASS, cu_config, make_oracle, make_sim

pytestmark = pytest.mark.gpu

EV = 1.602176634e-19 / (1.66053906892e-27 * 1.0e4)


def _dimers(reps, lo, hi, seed=3):
    """Boxes of two atoms each, `lo` to `hi` apart along x; and their distances"""
    from exastamp_amd import inputs
    d = np.exp(inputs.rng(seed).uniform(np.log(lo), np.log(hi), size=reps))
    r = np.full((reps, 2, 3), 4.0)
    r[:, 1, 0] += d
    d = r[:, 1, 0] - r[:, 0, 0]
    r = r.reshape(-1, 3)
    cfg = inputs.Config(r, np.zeros_like(r), np.zeros(2 * reps, np.uint8), np.zeros((reps, 3)),
                        np.full((reps, 3), 40.0), (1, 1, 1), np.repeat(np.arange(reps, dtype=np.uint16), 2))
    return cfg, d


def test_distance_and_its_reciprocal():
    """The FP64 EAM passes on tables that show them: rho(r) = r, so rho_i is the distance
    (three roundings of numbers up to 16, and of the knot fraction: 3e-15); r phi(r) = 1
    eV A, so ep is half the reciprocal (1.5 ulp and two roundings: 6e-16 relative)."""
    from exastamp_amd.potentials import SetflTables
    n, dr = 64, 0.25
    tab = SetflTables(["Cu"], [29], [CU_MASS], [3.6], ["fcc"], 5, 1.0, n, dr, 12.0, np.zeros((1, 5)),
                      np.arange(n)[None, :] * dr, np.ones((1, n)))
    cfg, d = _dimers(30000, 0.02, 11.9)
    sim = make_sim(cfg, [CU_MASS])
    sim.eam_alloy_init(tab)
    sim.chunk_neighbors(rcut_max=12.0, rcut_inc=0.3)
    sim.zero_force_energy()
    sim.eam_alloy_force(rcut=12.0, eam_rho2emb=False, eam_force=False)
    r = np.sqrt((d * d).astype(np.longdouble))
    rho = sim.rho_dEmb().reshape(-1, 2)
    assert np.array_equal(rho[:, 0], rho[:, 1]) and np.abs(rho[:, 0] - r).max() <= 3e-15
    sim.zero_force_energy()
    sim.eam_alloy_force(rcut=12.0, trigger_thermo_state=True)
    ep = sim.ep().reshape(-1, 2)
    want = np.longdouble(0.5) * np.longdouble(EV) / r
    assert np.array_equal(ep[:, 0], ep[:, 1]) and np.abs(ep[:, 0] / want - 1).max() <= 6e-16


def test_reciprocal_of_the_squared_distance():
    """The FP64 LJ force, whose roundings past 1/d2 are reproduced here: the reciprocal is
    within an ulp of the division, which the force (at these distances about the fourth
    power of it) shows as 1.2e-15 at most."""
    cfg, d = _dimers(30000, 2.0, 11.9, seed=4)
    sim = make_sim(cfg, [CU_MASS])
    sim.chunk_neighbors(rcut_max=12.0, rcut_inc=0.3)
    sim.zero_force_energy()
    sim.lj_compute_force(parameters={"epsilon": 1.0, "sigma": 1.0}, rcut=12.0)
    f = sim.accelerations().reshape(-1, 2, 3)  # forces: force_to_accel has not run
    ir2 = 1.0 / (d * d)
    s6 = ir2 * ir2 * ir2
    want = d * (-24.0 * (2.0 * (s6 * s6) - s6) * ir2)
    assert np.array_equal(f[:, 0], -f[:, 1]) and not f[:, :, 1:].any()
    assert np.abs(f[:, 0, 0] / want - 1.0).max() <= 1.2e-15


@pytest.mark.parametrize("atoms", ["400", None])  # bricks of many atoms; small ones, 16 lanes an atom
@pytest.mark.parametrize("species", [1, 2])
def test_odd_atom_counts_fp64(monkeypatch, species, atoms):
    """Clusters of 1 to 200 atoms, one to a box: the last atom of a brick without a
    neighbour lane, lists of 0 to 50 entries side by side.  Against the global list, whose
    lanes load their rows alone: 1e-10 of the rms, as for every order of the sums."""
    from exastamp_amd import inputs
    g = inputs.rng(12)
    sites = inputs.fcc(4, 4, 4, 3.6) + 0.7
    ks = list(range(1, 34)) + [63, 64, 65, 127, 129, 130, 191, 193, 200]
    r = np.concatenate([sites[g.permutation(len(sites))[:k]] for k in ks])
    r = r + g.normal(scale=0.05, size=r.shape)
    t = g.integers(0, species, size=len(r)).astype(np.uint8)
    cfg = inputs.Config(r, np.zeros_like(r), t, np.zeros((len(ks), 3)), np.full((len(ks), 3), 36.0), (1, 1, 1),
                        np.repeat(np.arange(len(ks), dtype=np.uint16), ks))
    tab = cu_tables(500) if species == 1 else cuni_tables(500)
    out = []
    for kind in ("block", "global"):
        for k in ("XSMD_LIST", "XSMD_BLOCK_ATOMS"):
            monkeypatch.delenv(k, raising=False)
        if kind == "global":
            monkeypatch.setenv("XSMD_LIST", "global")
        elif atoms:
            monkeypatch.setenv("XSMD_BLOCK_ATOMS", atoms)
        sim = make_sim(cfg, [CU_MASS, 58.693][:species])
        sim.eam_alloy_init(tab)
        sim.chunk_neighbors(rcut_max=tab.rc, rcut_inc=0.3)
        info = sim.list_info()
        assert info["kind"] == kind and (kind == "global" or not atoms or info["central_max"] > 128)
        sim.zero_force_energy()
        sim.eam_alloy_force(rcut=tab.rc, trigger_thermo_state=True, compute_virial=True)
        out.append((sim.accelerations(), sim.ep(), sim.virial(), sim.rho_dEmb()))
    for x, y in zip(*out):
        assert np.abs(x - y).max() <= 1e-10 * np.sqrt((y ** 2).mean())


@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1])
def test_cell_sort_around_its_one_kernel_form(oracle_mod, n):
    """Order of the sorted atoms, and that their data moved with them (exact)."""
    from exastamp_amd import inputs
    c = cu_config((64, 64, 33), jitter=0.02, seed=8)
    pick = inputs.rng(9).permutation(c.n)[:n]  # ids in no spatial order
    cfg = inputs.Config(c.r[pick], c.v[pick], c.type[pick], c.lo, c.hi)
    sim, o = make_sim(cfg, [CU_MASS]), make_oracle(oracle_mod, cfg, [CU_MASS])
    sim.chunk_neighbors(rcut_max=3.0, rcut_inc=0.3)
    o.build_neighbors(3.0, 0.3)
    assert np.array_equal(sim.order(), o.order())
    r, v = sim.state()
    assert np.array_equal(v, cfg.v) and np.array_equal(r, o.state()["r"])


@pytest.mark.parametrize("n", [5, 6, 9])
def test_adjoint_smallest_tables(monkeypatch, n):
    """Tables of 5 and 6 knots, where the special slopes at both ends overlap: FP64 adjoint
    against autograd, 1e-10 of the largest gradient of a table.  Some densities lie past
    tables as coarse as these, where F goes on with its last slope."""
    from exastamp_amd import inputs, units
    spline = sweeps._spline
    monkeypatch.setattr(sweeps, "_spline", lambda f, s, x, d: spline(f, s, x, d) +
                        s[-1] * (x / d - (len(f) - 1)).clamp(min=0.0))
    tab = cu_tables(n)
    cfg = inputs.lattice_config((3, 3, 3), 3.615, [CU_MASS], jitter=0.08, seed=6)
    g = inputs.rng(9)
    gF, gE = g.standard_normal((cfg.n, 3)), g.standard_normal(1)
    want, sizes = sweeps._reference(cfg, tab, gF, gE, ~0, None)
    sim = make_sim(cfg, [CU_MASS])
    sim.eam_alloy_init(tab)
    sim.chunk_neighbors(rcut_max=tab.rc, rcut_inc=0.3)
    sim.zero_force_energy()
    sim.eam_alloy_force(rcut=tab.rc, trigger_thermo_state=True)
    got = sim.eam_adjoint(gF / units.EV, gE / units.EV)
    for k, size in enumerate(sizes):
        a = sum(sizes[:k])
        assert np.abs(got[a:a + size] - want[a:a + size]).max() <= 1e-10 * np.abs(want[a:a + size]).max()
