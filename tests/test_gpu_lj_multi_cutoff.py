"""lj_multi_force at a pair's cutoff: a pair counts when r <= rcut, also where the square of
rcut rounds below d2 = r^2, and when a pair of species with a longer cutoff does not
interact (epsilon 0).  Dyadic displacements, so d2 is exact; the force against the
formula in FP64 (s^6 within 7 roundings, s^12 within 14, their difference at most four
times smaller than they are, on both sides: 1e-14 relative)."""
import math

import numpy as np
import pytest

from test_gpu_parity import make_sim

pytestmark = pytest.mark.gpu

MASSES = [65.38, 63.546]
EPS, SIG = 300.0, 2.4


@pytest.mark.parametrize("kind", ["block", "global"])
@pytest.mark.parametrize("long_pair", [True, False])
@pytest.mark.parametrize("dx,dy", [(2.125, 2.125), (2.1875, 2.25), (2.1875, 2.375), (3.0, 2.0)])
def test_pair_at_its_cutoff(monkeypatch, kind, long_pair, dx, dy):
    from exastamp_amd import inputs
    if kind == "global":
        monkeypatch.setenv("XSMD_LIST", "global")
    else:
        monkeypatch.delenv("XSMD_LIST", raising=False)
    d2 = dx * dx + dy * dy
    rc = math.sqrt(d2)
    r = np.array([[4.0, 4.0, 4.0], [4.0 + dx, 4.0 + dy, 4.0]])
    cfg = inputs.Config(r, np.zeros_like(r), np.array([0, 1], np.uint8), np.zeros((1, 3)), np.full((1, 3), 24.0))
    s6 = (SIG * SIG / d2) ** 3
    want = -24.0 * EPS * (2.0 * s6 * s6 - s6) / d2 * np.array([dx, dy, 0.0])
    for cut, inside in ((rc, True), (math.nextafter(rc, 0.0), False)):
        sim = make_sim(cfg, MASSES, ["Zn", "Cu"])
        sim.chunk_neighbors(rcut_max=6.0, rcut_inc=0.5)
        assert sim.list_info()["kind"] == kind
        sim.zero_force_energy()
        pairs = [{"type_a": "Zn", "type_b": "Cu", "rcut": cut, "parameters": {"epsilon": EPS, "sigma": SIG}}]
        sim.lj_multi_force(rcut=6.0 if long_pair else cut, parameters=pairs,
                           common_parameters={"epsilon": 0.0, "sigma": 0.0})
        f = sim.accelerations()  # forces: force_to_accel has not run
        assert np.array_equal(f[0], -f[1])
        assert np.abs(f[0] - (want if inside else 0.0)).max() <= 1e-14 * np.abs(want).max()
