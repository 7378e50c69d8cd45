"""Timed cases of the framework: what a molecular-dynamics or table-fitting program
has it do, through Simulation (exastamp_amd.operators) and the fitting functions
(exastamp_amd.fitting).

    listed()             the cases, as dicts of plain values
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call (inputs, loaded system)
    run(state)           one pass through the public entry points, and its outputs
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    the outputs of run in 64 bits, from plain numpy and torch

Kinds of case:
    point   one configuration evaluated: list build, forces, energies, virial
    md      md_run for `steps` NVE steps from the prepared state, then what the program
            keeps: the atoms' positions and velocities (`frame`), or the forces on the
            device, and the thermodynamic state every `sample` steps
    loop    the NVE step operator by operator, as a deck's scheme runs it
    fit     forces and energies of a configuration or a batch of them for table knots on
            the GPU, the fitting loss, and its gradient with respect to the knots

The mixed form computes pairs in single precision, so its outputs are kept in single
precision; the FP64 form's stay in double.
"""
import ctypes
import math

import numpy as np
import torch

from exastamp_amd.fitting import EamForcesEnergies, fit_loss
from exastamp_amd.inputs import Config
from exastamp_amd.operators import Simulation
from exastamp_amd.potentials import SetflTables

# internal units: Angstrom, Dalton, picosecond (energy Da.A^2/ps^2)
DALTON = 1.66053906892e-27
EV = 1.602176634e-19 / (DALTON * 1e4)
JOULE = 1.0 / (DALTON * 1e4)
KB = 1.380649e-23 / (DALTON * 1e4)

# Materials: the argon, copper, copper/nickel configurations of the benchmark, and the
# copper/zinc Lennard-Jones and tantalum Johnson decks of the tests.
MATERIALS = {
    "lj": dict(species=[("Ar", 39.948)], basis="fcc", a=5.26, T=100.0, jitter=0.1, rc=8.5, skin=0.3, dt=0.002),
    "ljmix": dict(species=[("Cu", 63.546), ("Zn", 65.38)], basis="fcc", a=5.0, T=300.0, jitter=0.1, rc=8.0, skin=1.0,
                  dt=0.001),
    "eam": dict(species=[("Cu", 63.546)], basis="fcc", a=3.615, T=600.0, jitter=0.05, rc=4.95, skin=0.3, dt=0.001),
    "alloy": dict(species=[("Cu", 63.546), ("Ni", 58.693)], basis="fcc", a=3.57, T=300.0, jitter=0.05, rc=4.95,
                  skin=0.3, dt=0.001),
    "johnson": dict(species=[("Ta", 180.95)], basis="bcc", a=3.3, T=300.0, jitter=0.05, rc=6.1, skin=1.0, dt=0.001),
}
BASIS = {
    "fcc": ((0.25, 0.25, 0.25), (0.75, 0.75, 0.25), (0.75, 0.25, 0.75), (0.25, 0.75, 0.75)),
    "bcc": ((0.25, 0.25, 0.25), (0.75, 0.75, 0.75)),
}
LJ_AR = {"epsilon": 0.0104 * EV, "sigma": 3.4}
# lj_multi_force of the Cu/Zn deck: Cu-Cu does not interact
LJ_MIX = [("Zn", "Zn", 6.10, 2.522e-20 * JOULE, 2.44), ("Cu", "Zn", 5.89, 4.853e-20 * JOULE, 2.36)]
JOHNSON_TA = {
    "re": 2.860082, "fe": 3.08634 * EV, "rhoe": 33.787168 * EV, "alpha": 8.489528, "beta": 4.527748,
    "A": 0.611679 * EV, "B": 1.032101 * EV, "kappa": 0.176977, "lambda": 0.353954, "Fn0": -5.103845 * EV,
    "Fn1": -0.405524 * EV, "Fn2": 1.112997 * EV, "Fn3": -3.585325 * EV, "F0": -5.14 * EV, "F1": 0.0,
    "F2": 1.640098 * EV, "F3": 0.221375 * EV, "Fo": -5.141526 * EV, "eta": 0.848843 * EV,
}
FIT_WEIGHT = 0.1


def _case(name, kind, pot, cells, mixed=False, steps=0, sample=0, frame=False, new=False, sym=False, nconf=1,
          knots=0):
    nx, ny, nz = cells
    c = dict(kind=kind, pot=pot, nx=nx, ny=ny, nz=nz, mixed=mixed, steps=steps, sample=sample, frame=frame, new=new,
             sym=sym, nconf=nconf, knots=knots)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # a new small configuration each time, as when a data set is evaluated: load it,
        # build its list, read forces, energies and virials back (864 atoms)
        _case("point_eam_864", "point", "eam", (6, 6, 6), new=True, frame=True),
        # the regression-size argon run: 4000 atoms, every launch and wait shows
        _case("md_lj_4k", "md", "lj", (10, 10, 10), steps=100, sample=10, frame=True),
        # an ordinary mid-size run on a ragged box, single-precision pairs
        _case("md_eam_50k_mixed", "md", "eam", (23, 29, 19), mixed=True, steps=100, sample=10, frame=True),
        # the half-million-atom double-precision run, one frame at its end
        _case("md_eam_500k", "md", "eam", (50, 50, 50), steps=100, sample=50, frame=True),
        # the million-atom argon benchmark
        _case("md_lj_1M_mixed", "md", "lj", (64, 64, 64), mixed=True, steps=50, sample=50),
        # the headline benchmark's system: 8.39 M copper atoms
        _case("md_eam_8M_mixed", "md", "eam", (128, 128, 128), mixed=True, steps=50, sample=50),
        # a deck's step, operator by operator: two species, vacancies, a free surface
        _case("loop_alloy_130k", "loop", "alloy", (32, 32, 32), steps=10, sample=10),
        # multi-species Lennard-Jones operator on a ragged box, energies and virial
        _case("point_ljmix_136k", "point", "ljmix", (37, 29, 31)),
        # Newton-symmetric EAM operator, as decks with eam_symmetry ask for
        _case("point_eam_sym_256k", "point", "eam", (40, 40, 40), sym=True),
        # analytic Johnson operator, tantalum
        _case("point_johnson_128k", "point", "johnson", (40, 40, 40)),
        # fitting steps: a batch of small boxes, and one large two-species slab
        _case("fit_batch_64x864", "fit", "eam", (6, 6, 6), nconf=64, knots=500),
        _case("fit_slab_1M", "fit", "alloy", (64, 64, 64), knots=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, atoms, per_cell, least):
    """Ragged cell counts of a box with about `atoms` atoms."""
    edge = (atoms / per_cell) ** (1.0 / 3.0)
    return tuple(max(least, int(round(edge * rng.uniform(0.75, 1.3)))) for _ in range(3))


def draw(rng):
    k = rng.randrange(6)
    if k == 0:  # runs of every size, both forms
        pot = rng.choice(["lj", "eam"])
        atoms = _log_int(rng, 3000, 1500000)
        steps = max(20, min(100, int(6e6 / atoms)))
        return _case(None, "md", pot, _box(rng, atoms, 4, 7), mixed=rng.random() < 0.5, steps=steps,
                     sample=rng.choice([10, steps]), frame=atoms < 200000)
    if k == 1:  # new configurations
        return _case(None, "point", rng.choice(["eam", "lj"]), _box(rng, _log_int(rng, 800, 60000), 4, 6), new=True,
                     frame=True)
    if k == 2:  # operators on a loaded system
        pot = rng.choice(["ljmix", "eam", "lj", "johnson"])
        return _case(None, "point", pot, _box(rng, _log_int(rng, 8000, 800000), 2 if pot == "johnson" else 4, 8),
                     mixed=pot != "johnson" and rng.random() < 0.3, sym=pot == "eam" and rng.random() < 0.4)
    if k == 3:  # operator by operator
        return _case(None, "loop", rng.choice(["alloy", "eam", "lj"]), _box(rng, _log_int(rng, 8000, 800000), 4, 8),
                     mixed=rng.random() < 0.5, steps=10, sample=10)
    if k == 4:  # batches of small boxes
        n = rng.randint(6, 8)
        return _case(None, "fit", "eam", (n, n, n), nconf=_log_int(rng, 4, 96), knots=rng.choice([400, 500, 1000]))
    return _case(None, "fit", "alloy", _box(rng, _log_int(rng, 20000, 1000000), 4, 8), knots=rng.choice([1000, 2000]))


# --- inputs ---------------------------------------------------------------------


def _tables(pot, knots):
    """Setfl tables of the embedded-atom materials: exponential densities, Morse pair
    terms, a square-root and quadratic embedding, tapered to zero at the cutoff."""
    n, rc = knots or (5000 if pot == "eam" else 2000), 4.95
    els = [dict(a=3.615, beta=6.0, E0=2.6, B=0.6, D=0.18, alpha=1.55, r0=2.97136, z=29, m=63.546)]
    if pot == "alloy":
        els.append(dict(a=3.52, beta=6.3, E0=2.9, B=0.7, D=0.2, alpha=1.6, r0=2.89409, z=28, m=58.693))
    dr = rc / (n - 1)
    r = np.arange(n) * dr
    x = np.clip(r - (rc - 1.0), 0.0, 1.0)
    taper = 1.0 - x ** 3 * (10.0 - 15.0 * x + 6.0 * x * x)
    shells = ((0.5, 12), (1.0, 6), (1.5, 24))  # FCC neighbours: distance^2 / a^2, count
    rho, phi, rho_e = [], [], []
    for e in els:
        f = np.exp(-e["beta"] * (r * math.sqrt(2.0) / e["a"] - 1.0)) * taper
        rho.append(f)
        rho_e.append(sum(c * float(np.interp(math.sqrt(s) * e["a"], r, f)) for s, c in shells))
        y = np.exp(-e["alpha"] * (r - e["r0"]))
        phi.append(e["D"] * (y * y - 2.0 * y) * taper)
    drho = 2.0 * max(rho_e) / (n - 1)
    frho = []
    for e, re in zip(els, rho_e):
        q = np.arange(n) * drho / re
        frho.append(-e["E0"] * np.sqrt(q) + e["B"] * (q - 1.0) ** 2)
    z2r = [r * 0.5 * (phi[i] + phi[j]) for i in range(len(els)) for j in range(i + 1)]
    names = [s for s, _ in MATERIALS[pot]["species"]]
    return SetflTables(names, [e["z"] for e in els], [e["m"] for e in els], [e["a"] for e in els],
                       ["fcc"] * len(els), n, drho, n, dr, rc, np.array(frho), np.array(rho), np.array(z2r))


def _lattice(basis, cells, a):
    nx, ny, nz = cells
    g = np.empty((nz, ny, nx, len(BASIS[basis]), 3))
    for b, o in enumerate(BASIS[basis]):
        g[..., b, 0] = ((np.arange(nx) + o[0]) * a)[None, None, :]
        g[..., b, 1] = ((np.arange(ny) + o[1]) * a)[None, :, None]
        g[..., b, 2] = ((np.arange(nz) + o[2]) * a)[:, None, None]
    return g.reshape(-1, 3)


def _velocities(g, mass, T):
    v = g.standard_normal((len(mass), 3)) * np.sqrt(KB * T / mass)[:, None]
    return v - (mass[:, None] * v).sum(0) / mass.sum()


def _config(case, seed):
    m = MATERIALS[case["pot"]]
    g = np.random.Generator(np.random.SFC64([seed, 77]))
    cells = (case["nx"], case["ny"], case["nz"])
    masses = np.array([w for _, w in m["species"]])
    if case["nconf"] > 1:  # boxes of their own strain (+-3 %) and temperature (300-1500 K)
        rs, his = [], []
        for _ in range(case["nconf"]):
            a = m["a"] * (1.0 + g.uniform(-0.03, 0.03))
            r = _lattice(m["basis"], cells, a)
            rs.append(r + g.standard_normal(r.shape) * 0.05 * math.sqrt(g.uniform(300.0, 1500.0) / 300.0))
            his.append([c * a for c in cells])
        r = np.concatenate(rs)
        rep = np.repeat(np.arange(case["nconf"], dtype=np.uint16), len(rs[0]))
        return Config(r, np.zeros_like(r), np.zeros(len(r), np.uint8), np.zeros((case["nconf"], 3)), np.array(his),
                      (1, 1, 1), rep)
    r = _lattice(m["basis"], cells, m["a"])
    hi = np.array([[c * m["a"] for c in cells]])
    t = np.zeros(len(r), np.uint8)
    periodic = (1, 1, 1)
    if case["pot"] == "ljmix":
        t[1::2] = 1
    if case["pot"] == "alloy":  # half of the sites each, 1 % vacancies, vacuum on both sides along z
        t = (g.random(len(r)) < 0.5).astype(np.uint8)
        keep = np.ones(len(r), bool)
        keep[g.permutation(len(r))[:len(r) // 100]] = False
        r, t = r[keep], t[keep]
        r[:, 2] += 10.0
        hi[0, 2] += 20.0
        periodic = (1, 1, 0)
    r += g.standard_normal(r.shape) * m["jitter"]
    return Config(r, _velocities(g, masses[t], m["T"]), t, np.zeros((1, 3)), hi, periodic)


def _theta(tab, seed):
    """The knots a fitting program starts from: 2 % off the tables that made its targets."""
    t = tab.theta()
    g = np.random.Generator(np.random.SFC64([seed, 78]))
    return t * (1.0 + g.uniform(-0.02, 0.02, t.size))


def _targets(cfg, seed):
    g = np.random.Generator(np.random.SFC64([seed, 79]))
    n = np.bincount(cfg.rep) if cfg.rep is not None else np.array([cfg.n])
    return g.standard_normal((cfg.n, 3)) * 0.5, (-3.5 + 0.05 * g.standard_normal(len(n))) * n, n.astype(np.float64)


# --- the calls ------------------------------------------------------------------


def _forces(s, c):
    """The potential's operator with energies and virial, for the current list."""
    sim, rc = s["sim"], s["m"]["rc"]
    if c["pot"] == "lj":
        sim.lj_compute_force(parameters=LJ_AR, rcut=rc, mixed=c["mixed"])
    elif c["pot"] == "ljmix":
        sim.lj_multi_force(rcut=rc, mixed=c["mixed"], parameters=[
            {"type_a": a, "type_b": b, "rcut": r, "parameters": {"epsilon": e, "sigma": g}} for a, b, r, e, g in LJ_MIX])
    elif c["pot"] == "johnson":
        sim.johnson_force(rcut=rc, parameters=JOHNSON_TA, compute_virial=True)
    else:
        sim.eam_alloy_force(rcut=rc, trigger_thermo_state=True, compute_virial=True, mixed=c["mixed"],
                            eam_symmetry=c["sym"])


def _device_forces(sim):
    """Forces (n, 3) in eV/A on the device."""
    F = torch.empty((sim.n, 3), dtype=torch.float64, device="cuda")
    E = torch.empty(sim.cfg.nrep, dtype=torch.float64, device="cuda")
    sim.ctx.xs_forces_energies_dev(ctypes.c_void_p(F.data_ptr()), ctypes.c_void_p(E.data_ptr()), 1.0 / EV)
    return F


def _kept(out, mixed):
    if not mixed:
        return out
    return {k: v.float() if isinstance(v, torch.Tensor) else v.astype(np.float32) for k, v in out.items()}


def prepare(case, seed):
    m = MATERIALS[case["pot"]]
    cfg = _config(case, seed)
    sim = Simulation(0)
    sim.species(m["species"])
    s = dict(sim=sim, case=case, m=m, cfg=cfg)
    if not case["new"]:
        sim.set_config(cfg)
    if case["pot"] in ("eam", "alloy"):
        tab = _tables(case["pot"], case["knots"])
        sim.eam_alloy_init(tab)
    elif case["pot"] == "lj":
        sim.lj_parameters(LJ_AR, m["rc"])
    if case["kind"] != "fit" and not case["frame"]:
        # forces stay on the device: the library works on torch's stream
        sim.ctx.xs_ctx_set_stream(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if case["kind"] == "loop":
        sim.chunk_neighbors(rcut_max=m["rc"], rcut_inc=m["skin"])
        sim.zero_force_energy()
        _forces(s, case)
        sim.force_to_accel()
    if case["kind"] == "fit":
        sim.chunk_neighbors(rcut_max=m["rc"], rcut_inc=m["skin"])
        Ft, Et, n = _targets(cfg, seed)
        s["theta"] = torch.tensor(_theta(tab, seed), device="cuda", requires_grad=True)
        s["Ft"], s["Et"], s["n"] = (torch.tensor(x, device="cuda") for x in (Ft, Et, n))
    return s


def run(s):
    c, m, sim = s["case"], s["m"], s["sim"]
    if c["kind"] == "fit":
        s["theta"].grad = None
        F, E = EamForcesEnergies.apply(s["theta"], sim)
        loss = fit_loss(F, E, s["Ft"], s["Et"], s["n"], FIT_WEIGHT)
        loss.backward()
        return dict(F=F.detach(), E=E.detach(), loss=loss.detach(), grad=s["theta"].grad)
    if c["kind"] == "md":
        _, th = sim.md_run("lj" if c["pot"] == "lj" else "eam", c["steps"], m["dt"], m["rc"], m["skin"],
                           mixed=c["mixed"], thermo_every=c["sample"])
        out = dict(thermo=np.stack([t.raw for t in th]))
        if c["frame"]:
            out["r"], out["v"] = sim.state()
        else:
            out["F"] = _device_forces(sim)
        return _kept(out, c["mixed"])
    if c["kind"] == "loop":
        for _ in range(c["steps"]):
            sim.push_f_v_r(m["dt"])
            sim.push_f_v(m["dt"], 0.5)
            if sim.particle_displ_over(0.5 * m["skin"]):
                sim.chunk_neighbors(rcut_max=m["rc"], rcut_inc=m["skin"])
            sim.zero_force_energy()
            _forces(s, c)
            sim.force_to_accel()
            sim.push_f_v(m["dt"], 0.5)
        return _kept(dict(thermo=sim.simulation_thermodynamic_state().raw, F=_device_forces(sim)), c["mixed"])
    if c["new"]:
        sim.set_config(s["cfg"])
    sim.chunk_neighbors(rcut_max=m["rc"], rcut_inc=m["skin"])
    sim.zero_force_energy()
    _forces(s, c)
    sim.force_to_accel()
    out = dict(thermo=sim.simulation_thermodynamic_state().raw)
    if c["frame"]:
        out["F"], out["ep"], out["virial"] = sim.forces(), sim.ep(), sim.virial()
    else:
        out["F"] = _device_forces(sim)
    return _kept(out, c["mixed"])


def work(case):
    m = MATERIALS[case["pot"]]
    n = case["nx"] * case["ny"] * case["nz"] * len(BASIS[m["basis"]]) * case["nconf"]
    pairs = n * len(BASIS[m["basis"]]) / m["a"] ** 3 * 4.0 / 3.0 * math.pi * m["rc"] ** 3
    per_pair = {"lj": 22, "ljmix": 22, "eam": 70, "alloy": 70, "johnson": 150}[case["pot"]]
    if case["kind"] == "md":  # a step reads and writes positions and velocities
        return dict(bytes=96.0 * n * case["steps"], flops=pairs * per_pair * (case["steps"] + 1))
    if case["kind"] == "loop":
        return dict(bytes=96.0 * n * case["steps"], flops=pairs * (per_pair + 30) * case["steps"])
    if case["kind"] == "fit":  # positions, targets; forces written; the gradient sweep evaluates each pair again
        return dict(bytes=(24.0 + 24.0 + 24.0) * n, flops=pairs * (per_pair + 120.0))
    return dict(bytes=(24.0 + 24.0 + (80.0 if case["frame"] else 0.0)) * n, flops=pairs * (per_pair + 30))


# --- the same in 64 bits, plain torch ---------------------------------------------


def _neighbours(r, L, periodic, reach):
    """Padded neighbour matrix (n, k): every atom within `reach` (minimum image along the
    periodic axes), the atom itself as padding."""
    n, dev = r.shape[0], r.device
    per = torch.tensor(periodic, dtype=torch.bool, device=dev)
    lo = torch.where(per, torch.zeros(3, dtype=r.dtype, device=dev), r.min(0).values)
    ext = torch.where(per, L, r.max(0).values - lo + 1e-9)
    x = r - lo
    x = torch.where(per, x - torch.floor(x / ext) * ext, x)
    nc = torch.clamp((ext / reach).long(), min=1)
    if bool((per & (nc < 3)).any()):
        raise ValueError("box too small for the minimum image")
    c = torch.minimum((x / ext * nc).long(), nc - 1)
    key = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
    ncell = int(nc.prod())
    count = torch.bincount(key, minlength=ncell)
    order = torch.argsort(key, stable=True)
    start = torch.cumsum(count, 0) - count
    fill = int(count.max())
    table = torch.full((ncell + 1, fill), -1, dtype=torch.int64, device=dev)  # the last row: no cell
    ks = key[order]
    table[ks, torch.arange(n, device=dev) - start[ks]] = order
    off = torch.tensor([[i, j, k] for k in (-1, 0, 1) for j in (-1, 0, 1) for i in (-1, 0, 1)], device=dev)
    rows, kmax, parts = max(1, int(3e7 / (27 * fill))), 0, []
    for a in range(0, n, rows):
        i = torch.arange(a, min(n, a + rows), device=dev)
        q = c[i][:, None, :] + off[None]
        w = torch.where(per, q % nc, q)
        ok = ((w >= 0) & (w < nc)).all(2)
        cell = torch.where(ok, (w[..., 2] * nc[1] + w[..., 1]) * nc[0] + w[..., 0], ncell)
        j = table[cell].reshape(len(i), -1)
        d = _displacement(r, L, per, i, j.clamp(min=0))
        near = (j >= 0) & (j != i[:, None]) & ((d * d).sum(2) < reach * reach)
        k = near.sum(1)
        kmax = max(kmax, int(k.max()))
        parts.append((i, k, j[near]))
    out = torch.arange(n, device=dev)[:, None].repeat(1, kmax)
    for i, k, j in parts:
        at = torch.arange(len(j), device=dev) - torch.repeat_interleave(torch.cumsum(k, 0) - k, k)
        out[torch.repeat_interleave(i, k), at] = j
    return out


def _displacement(r, L, per, i, j):
    d = r[j] - r[i][:, None, :]
    return d - torch.where(per, torch.round(d / L), torch.zeros_like(L)) * L


def _spline(f):
    """Value coefficients (..., n, 4) of the setfl spline through knots f (..., n)."""
    s = torch.cat([(f[..., 1] - f[..., 0])[..., None], 0.5 * (f[..., 2] - f[..., 0])[..., None],
                   ((f[..., :-4] - f[..., 4:]) + 8.0 * (f[..., 3:-1] - f[..., 1:-3])) / 12.0,
                   0.5 * (f[..., -1] - f[..., -3])[..., None], (f[..., -1] - f[..., -2])[..., None]], -1)
    dv, z = f[..., 1:] - f[..., :-1], torch.zeros_like(f[..., :1])
    b = torch.cat([3.0 * dv - 2.0 * s[..., :-1] - s[..., 1:], z], -1)
    a = torch.cat([s[..., :-1] + s[..., 1:] - 2.0 * dv, z], -1)
    return torch.stack([a, b, s, f], -1)


def _at(coef, table, x, rdx):
    """Value and slope of spline `table` at x."""
    p = x * rdx
    m = torch.clamp(p.detach().long(), 0, coef.shape[1] - 2)
    p = torch.clamp(p - m, max=1.0)
    c = coef.reshape(-1, 4)[table * coef.shape[1] + m]
    return (((c[..., 0] * p + c[..., 1]) * p + c[..., 2]) * p + c[..., 3],
            ((3.0 * c[..., 0] * p + 2.0 * c[..., 1]) * p + c[..., 2]) * rdx)


class _Exact:
    """Energies, forces and virials of a material on a padded neighbour matrix."""

    def __init__(self, case, cfg, box, tab=None, theta=None):
        self.case, self.m = case, MATERIALS[case["pot"]]
        dev = torch.device("cuda")
        self.L = torch.tensor(box, dtype=torch.float64, device=dev)
        self.periodic = cfg.periodic
        self.per = torch.tensor(cfg.periodic, dtype=torch.bool, device=dev)
        self.type = torch.tensor(cfg.type.astype(np.int64), device=dev)
        self.mass = torch.tensor([w for _, w in self.m["species"]], dtype=torch.float64, device=dev)[self.type]
        if tab is not None:
            self.tab = tab
            t = theta if theta is not None else torch.tensor(tab.theta(), device=dev)
            nf, nr = tab.frho.size, tab.rhor.size
            self.F = _spline(t[:nf].reshape(tab.frho.shape))
            self.R = _spline(t[nf:nf + nr].reshape(tab.rhor.shape))
            self.Z = _spline(t[nf + nr:].reshape(tab.z2r.shape))

    def _chunks(self, n, k):
        rows = max(1, int(1.5e8 / k))
        return [(a, min(n, a + rows)) for a in range(0, n, rows)]

    def _pairs(self, r, nb, a, b):
        i = torch.arange(a, b, device=r.device)
        j = nb[a:b]
        d = _displacement(r, self.L, self.per, i, j)
        d2 = (d * d).sum(2)
        own = j == i[:, None]
        return i, j, d, torch.where(own, torch.ones_like(d2), d2), ~own & (d2 <= self.m["rc"] ** 2)

    def _lj(self, i, j, d2, on):
        m = self.m
        if self.case["pot"] == "lj":
            eps, sig, rc = LJ_AR["epsilon"], LJ_AR["sigma"], m["rc"]
        else:
            tab = torch.zeros((2, 2, 3), dtype=torch.float64, device=d2.device)
            tab[0, 0] = torch.tensor([0.0, 1.0, m["rc"]])
            for a, b, cut, e, s in LJ_MIX:
                x, y = ("Cu", "Zn").index(a), ("Cu", "Zn").index(b)
                tab[x, y] = tab[y, x] = torch.tensor([e, s, cut], dtype=torch.float64)
            eps, sig, rc = tab[self.type[i][:, None], self.type[j]].unbind(-1)
            on = on & (torch.sqrt(d2) <= rc)
        s6, c6 = (sig * sig / d2) ** 3, (sig / rc) ** 6
        e = 4.0 * eps * ((s6 * s6 - s6) - (c6 * c6 - c6))
        w = -24.0 * eps * (2.0 * s6 * s6 - s6) / d2
        return torch.where(on, e, 0.0 * e), torch.where(on, w, 0.0 * w)

    @staticmethod
    def _johnson_term(c, a, k, r):
        x = r / JOHNSON_TA["re"]
        num, s = c * torch.exp(-a * (x - 1.0)), x - k
        s19 = s ** 19
        den = 1.0 + s19 * s
        return num / den, (-a * num * den - num * 20.0 * s19) / (den * den) / JOHNSON_TA["re"]

    def _johnson_embed(self, rho):
        p, q = JOHNSON_TA, rho / JOHNSON_TA["rhoe"]
        t, u = q / 0.85 - 1.0, q - 1.0
        lo = p["Fn0"] + t * (p["Fn1"] + t * (p["Fn2"] + t * p["Fn3"]))
        dlo = (p["Fn1"] + t * (2.0 * p["Fn2"] + t * 3.0 * p["Fn3"])) / (0.85 * p["rhoe"])
        hi = p["F0"] + u * (p["F1"] + u * (p["F2"] + u * p["F3"]))
        dhi = (p["F1"] + u * (2.0 * p["F2"] + u * 3.0 * p["F3"])) / p["rhoe"]
        return torch.where(q < 0.85, lo, hi), torch.where(q < 0.85, dlo, dhi)

    def _functions(self, i, j, r):
        """rho into i and its slope, the slope of rho into j, phi and its slope."""
        if self.case["pot"] == "johnson":
            p = JOHNSON_TA
            rho, drho = self._johnson_term(p["fe"], p["beta"], p["lambda"], r)
            a, da = self._johnson_term(p["A"], p["alpha"], p["kappa"], r)
            b, db = self._johnson_term(p["B"], p["beta"], p["lambda"], r)
            return rho, drho, drho, a - b, da - db
        ti, tj, rdr = self.type[i][:, None], self.type[j], 1.0 / self.tab.dr
        rho, drho = _at(self.R, tj, r, rdr)
        back = drho if len(self.m["species"]) == 1 else _at(self.R, ti.expand_as(tj), r, rdr)[1]
        hi, lo = torch.maximum(ti.expand_as(tj), tj), torch.minimum(ti.expand_as(tj), tj)
        z, dz = _at(self.Z, hi * (hi + 1) // 2 + lo, r, rdr)
        return rho, drho, back, EV * z / r, EV * (dz - z / r) / r

    def _embed(self, rho):
        if self.case["pot"] == "johnson":
            return self._johnson_embed(rho)
        f, df = _at(self.F, self.type, rho, 1.0 / self.tab.drho)
        return EV * f, EV * df

    def forces(self, r, nb):
        """Forces, per-atom energies and virials."""
        n, k = nb.shape
        F = torch.empty((n, 3), dtype=torch.float64, device=r.device)
        ep = torch.empty(n, dtype=torch.float64, device=r.device)
        vir = torch.empty((n, 3, 3), dtype=torch.float64, device=r.device)
        eam = self.case["pot"] not in ("lj", "ljmix")
        if eam:
            rho = torch.empty(n, dtype=torch.float64, device=r.device)
            for a, b in self._chunks(n, k):
                i, j, d, d2, on = self._pairs(r, nb, a, b)
                v = self._functions(i, j, torch.sqrt(d2))[0]
                rho[a:b] = torch.where(on, v, 0.0 * v).sum(1)
            emb, slope = self._embed(rho)
        for a, b in self._chunks(n, k):
            i, j, d, d2, on = self._pairs(r, nb, a, b)
            if eam:
                x = torch.sqrt(d2)
                _, drho, back, phi, dphi = self._functions(i, j, x)
                w = (slope[i][:, None] * drho + slope[j] * back + dphi) / x
                e, w = torch.where(on, phi, 0.0 * phi), torch.where(on, w, 0.0 * w)
            else:
                e, w = self._lj(i, j, d2, on)
            f = w[..., None] * d
            F[a:b] = f.sum(1)
            ep[a:b] = 0.5 * e.sum(1) + (emb[a:b] if eam else 0.0)
            vir[a:b] = -0.5 * torch.bmm(f.transpose(1, 2).contiguous(), d)
        return F, ep, vir

    def thermo(self, v, ep, vir):
        k = torch.einsum("na,nb->ab", self.mass[:, None] * v, v)
        out = torch.cat([vir.sum(0).reshape(9), 0.5 * k.reshape(9), (self.mass[:, None] * v).sum(0),
                         0.5 * torch.diagonal(k), ep.sum()[None], self.mass.sum()[None]])
        return np.append(out.cpu().numpy(), float(len(ep)))

    def wrap(self, r):
        r = torch.where(self.per & (r < 0.0), r + self.L, r)
        return torch.where(self.per & (r >= self.L), r - self.L, r)


def _exact_fit(case, seed):
    cfg = _config(case, seed)
    tab = _tables(case["pot"], case["knots"])
    theta = torch.tensor(_theta(tab, seed), device="cuda", requires_grad=True)
    Ft, Et, n = (torch.tensor(x, device="cuda") for x in _targets(cfg, seed))
    grad, Fs, Es, loss = torch.zeros_like(theta), [], [], 0.0
    for k in range(case["nconf"]):
        at = np.arange(cfg.n) if cfg.rep is None else np.flatnonzero(cfg.rep == k)
        one = Config(cfg.r[at], cfg.v[at], cfg.type[at], cfg.lo[k:k + 1], cfg.hi[k:k + 1], cfg.periodic)
        x = _Exact(case, one, one.hi[0], tab, theta)
        r = torch.tensor(one.r, device="cuda", requires_grad=True)
        nb = _neighbours(r.detach(), x.L, x.periodic, x.m["rc"])
        i, j, d, d2, on = x._pairs(r, nb, 0, one.n)
        rho, _, _, phi, _ = x._functions(i, j, torch.sqrt(d2))
        e = x._embed(torch.where(on, rho, 0.0 * rho).sum(1))[0].sum() + 0.5 * torch.where(on, phi, 0.0 * phi).sum()
        F = -torch.autograd.grad(e, r, create_graph=True)[0] / EV
        E = e / EV
        part = ((F - Ft[torch.tensor(at, device="cuda")]) ** 2).sum() / (3 * cfg.n) \
            + FIT_WEIGHT * ((E - Et[k]) / n[k]) ** 2 / case["nconf"]
        grad += torch.autograd.grad(part, theta)[0]
        Fs.append(F.detach())
        Es.append(E.detach())
        loss = loss + part.detach()
    return dict(F=torch.cat(Fs), E=torch.stack(Es), loss=loss, grad=grad)


def exact(case, seed):
    if case["kind"] == "fit":
        return _exact_fit(case, seed)
    cfg, m = _config(case, seed), MATERIALS[case["pot"]]
    tab = _tables(case["pot"], case["knots"]) if case["pot"] in ("eam", "alloy") else None
    x = _Exact(case, cfg, cfg.hi[0], tab)
    r, v = torch.tensor(cfg.r, device="cuda"), torch.tensor(cfg.v, device="cuda")
    r = x.wrap(r)
    wide = 2.0 * m["skin"] if case["steps"] else 0.0  # neighbours kept beyond the cutoff between searches
    near, at = _neighbours(r, x.L, x.periodic, m["rc"] + wide), r.clone()
    F, ep, vir = x.forces(r, near)
    if case["kind"] == "point":
        out = dict(thermo=x.thermo(v, ep, vir), F=F / EV)
        if case["frame"]:
            out.update(F=F, ep=ep, virial=vir)
        return out
    ref, dt, acc, seen = r.clone(), m["dt"], F / x.mass[:, None], []
    if case["kind"] == "md":
        seen.append(x.thermo(v, ep, vir))
    for step in range(1, case["steps"] + 1):
        r = r + (v * dt + acc * (0.5 * dt * dt))
        v = v + acc * (0.5 * dt)
        if float(((r - ref) ** 2).sum(1).max()) > (0.5 * m["skin"]) ** 2:  # a new list: atoms return to the box
            r = x.wrap(r)
            ref = r.clone()
        d = r - at
        d = d - torch.where(x.per, torch.round(d / x.L), torch.zeros_like(x.L)) * x.L
        if float((d * d).sum(1).max()) > (0.5 * wide) ** 2:
            near, at = _neighbours(r, x.L, x.periodic, m["rc"] + wide), r.clone()
        F, ep, vir = x.forces(r, near)
        acc = F / x.mass[:, None]
        v = v + acc * (0.5 * dt)
        if case["kind"] == "md" and step % case["sample"] == 0:
            seen.append(x.thermo(v, ep, vir))
    if case["kind"] == "loop":
        return dict(thermo=x.thermo(v, ep, vir), F=F / EV)
    out = dict(thermo=np.stack(seen))
    out.update(dict(r=r, v=v) if case["frame"] else dict(F=F / EV))
    return out
