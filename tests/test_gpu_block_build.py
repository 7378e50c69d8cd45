"""The cell-block list build at the sizes where its pieces meet: candidates of a cell
that fill one or several register tiles or less than one wave, lists around the sorted
limit of 64 entries and past the first capacity estimate, cells with fewer, as many and
more atoms than one collection of lists, empty cells, one cell per axis.  The list
converted back equals the global build entry for entry (both are exact, so bit-exact),
and a brick list was built (it is not the global build compared with itself) wherever the
halo of a one-cell brick, 27 cells, fits the passes' 64 KB of LDS at 32 bytes an atom."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _config(n, box, seed, cluster=0.0):
    from exastamp_amd import inputs
    g = inputs.rng(seed)
    r = g.random((n, 3)) * np.asarray(box)
    if cluster > 0:  # half of the atoms crowded into one corner
        r[: n // 2] = g.random((n // 2, 3)) * cluster
    return inputs.Config(r, np.zeros((n, 3)), np.zeros(n, np.uint8), np.zeros((1, 3)), np.array([box], float))


def _lists(monkeypatch, kind, cfg, rcut):
    from exastamp_amd.operators import Simulation
    if kind == "global":
        monkeypatch.setenv("XSMD_LIST", "global")
    else:
        monkeypatch.delenv("XSMD_LIST", raising=False)
    sim = Simulation(0)
    sim.species([("Ar", 39.948)])
    sim.set_config(cfg)
    sim.chunk_neighbors(rcut_max=rcut, rcut_inc=0.3)
    out = sim.neighbors() + (sim.order(),)
    info = sim.list_info()
    sim.close()
    return out, info


@pytest.mark.parametrize("n,box,rcut,cluster", [
    (1, (12.0, 12.0, 12.0), 4.0, 0.0),          # one atom
    (700, (60.0, 55.0, 50.0), 4.0, 0.0),        # fewer than one atom per cell on average
    (4000, (40.0, 37.0, 43.0), 4.0, 0.0),       # about 5 per cell, one tile
    (6000, (36.0, 33.0, 30.0), 4.0, 0.0),       # about 13 per cell, lists around 64
    (3000, (26.0, 31.0, 22.0), 5.0, 0.0),       # about 25 per cell, several tiles
    (1500, (12.0, 12.0, 18.0), 5.7, 0.0),       # 125 per cell: the halo does not fit
    (900, (9.0, 9.0, 9.0), 4.0, 0.0),           # 112 per cell: likewise
    (300, (6.0, 6.0, 6.0), 4.0, 0.0),           # 300 in the one cell: likewise
    (1200, (16.5, 16.5, 16.5), 5.0, 0.0),       # 44 per cell, over 512 candidates
    (200, (9.0, 9.0, 9.0), 4.0, 0.0),           # two cells per axis, each neighbour seen through two images
    (40, (6.0, 6.0, 6.0), 4.0, 0.0),            # one cell: images of every atom on all sides
    (2400, (44.0, 44.0, 44.0), 4.0, 9.0),       # crowded corner: lists far beyond the mean-density estimate
])
def test_block_lists_equal_global(monkeypatch, n, box, rcut, cluster):
    cfg = _config(n, box, seed=n, cluster=cluster)
    glob, ginfo = _lists(monkeypatch, "global", cfg, rcut)
    blk, info = _lists(monkeypatch, "block", cfg, rcut)
    ncell = np.prod([max(1, int(x / (rcut + 0.3))) for x in box])
    fits = 27 * n / ncell * 32 < 60e3 or cluster > 0
    assert ginfo["kind"] == "global" and info["kind"] == ("block" if fits else "global")
    print(f"{n} atoms: longest list {glob[0].max()}, brick {info['brick']}, halo {info['halo_capacity']}")
    for x, y in zip(blk, glob):
        assert np.array_equal(x, y)


def test_tables_of_a_cluster_in_a_large_box(monkeypatch):
    """A dense cluster in a box of 600 k cells: the bricks' tables go with the atoms (3000
    atoms, at most 27 staging entries each and their padding), not with the number of
    bricks times the densest one (gigabytes here).  200 MB covers the per-cell arrays."""
    from exastamp_amd.operators import Simulation
    import ctypes as C
    cfg = _config(3000, (370.0, 365.0, 360.0), seed=7, cluster=13.0)
    glob, _ = _lists(monkeypatch, "global", cfg, 4.0)
    monkeypatch.delenv("XSMD_LIST", raising=False)
    sim = Simulation(0)
    sim.species([("Ar", 39.948)])
    sim.set_config(cfg)
    free = [C.c_size_t(0), C.c_size_t(0)]
    total = C.c_size_t(0)
    sim.ctx.xs_device_memory(C.byref(free[0]), C.byref(total))
    sim.chunk_neighbors(rcut_max=4.0, rcut_inc=0.3)
    sim.ctx.xs_device_memory(C.byref(free[1]), C.byref(total))
    assert sim.list_info()["kind"] == "block"
    blk = sim.neighbors() + (sim.order(),)
    sim.close()
    for x, y in zip(blk, glob):
        assert np.array_equal(x, y)
    assert free[0].value - free[1].value < 200e6
