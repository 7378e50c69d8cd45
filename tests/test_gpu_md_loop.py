"""The MD loop where it queues steps ahead of the rebuild test: a run continued with
XS_CONTINUE, a list without skin (every step rebuilds), and rebuild intervals that move
while steps are queued.  Two runs of the same steps differ only by the order their lists
are summed in, FP64 rounding at rms force 1e-15 grown over 40 steps: 1e-10 of the total
energy is far above that and far below the energy exchanged in a step."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RC, DT = 8.5, 0.002


def _sim(cells=7):
    from exastamp_amd import inputs
    from exastamp_amd.operators import Simulation
    g = inputs.rng(11)
    base = np.array([(0.25, 0.25, 0.25), (0.75, 0.75, 0.25), (0.75, 0.25, 0.75), (0.25, 0.75, 0.75)])
    grid = np.stack(np.meshgrid(*[np.arange(cells)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    r = ((grid + base).reshape(-1, 3)) * 5.26 + 0.1 * g.standard_normal((4 * cells ** 3, 3))
    v = 1.5 * g.standard_normal(r.shape)
    L = 5.26 * cells
    cfg = inputs.Config(r, v - v.mean(0), np.zeros(len(r), np.uint8), np.zeros((1, 3)), np.array([[L, L, L]]))
    sim = Simulation(0)
    sim.species([("Ar", 39.948)])
    sim.set_config(cfg)
    sim.lj_parameters({"epsilon": 100.0, "sigma": 3.4}, RC)
    return sim


def _run(sim, steps, skin, flags=0, every=1, fill=np.nan):
    from exastamp_amd import _lib
    out = np.full(27 * (steps // every + 1), fill)
    st = _lib.RunStats()
    sim.ctx.xs_md_run(_lib.XS_POT_LJ, steps, DT, RC, skin, flags, every, _lib.dptr(out), C.byref(st))
    return out.reshape(-1, 27), st


def _total(rows):
    return rows[:, 21:25].sum(1)


def test_continued_run_leaves_step_0():
    sim = _sim()
    whole, _ = _run(sim, 40, 0.3)
    sim.close()
    sim = _sim()
    first, _ = _run(sim, 15, 0.3)
    second, _ = _run(sim, 25, 0.3, flags=8, fill=-7.0)
    sim.close()
    assert (second[0] == -7.0).all()
    E = np.concatenate([_total(first), _total(second[1:])])
    assert np.abs(E - _total(whole)).max() <= 1e-10 * np.abs(_total(whole)).max()


@pytest.mark.parametrize("skin,every", [(0.0, 1), (0.0, 40), (0.05, 7), (1.0, 40)])
def test_rebuild_intervals(skin, every):
    sim = _sim()
    ref, _ = _run(sim, 40, 0.3)
    sim.close()
    sim = _sim()
    rows, st = _run(sim, 40, skin, every=every)
    r, v = sim.state()
    sim.close()
    assert np.isfinite(r).all() and np.isfinite(v).all()
    if skin == 0.0:
        assert st.rebuilds == 41
    want = _total(ref)[::every]
    assert np.abs(_total(rows) - want).max() <= 1e-10 * np.abs(want).max()
