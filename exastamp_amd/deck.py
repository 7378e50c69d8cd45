"""Runner for exaStamp YAML operator-graph decks, restricted to the force path.

exaStamp runs a simulation as a graph of named operators described in YAML
``.msp`` decks (data/config/main-config.msp and the files it includes; a user deck
overrides nodes by name).  This module reads such decks -- ``includes``, node
aliases, batches, blocks with ``rebind`` / ``body`` / ``loop`` / ``condition``,
``+name`` list appends, ``--set-a-b-c value`` overrides -- and executes the subset
of the graph this library implements: ``setup_system`` (species, particle types,
domain, FCC/BCC/SC ``lattice``, ``gaussian_noise_r/v``), ``init_parameters``
(``eam_alloy_init``), the NVE scheme (``verlet_first_half``,
``check_and_update_particles``, ``compute_all_forces_energy``,
``verlet_second_half``), the force operators (``lj_compute_force``,
``eam_alloy_force`` with its pass flags), ``chunk_neighbors`` and the
thermodynamic state on the screen/file frequencies of ``global``.

The default graph below restates the node names and the control flow of the
reference's default NVE simulation (main-config.msp:145-170,232-255,
config_numerical_schemes.msp:8-52, config_move_particles.msp:17-152,
config_globals.msp:5-29) for that subset; a deck overrides it exactly as it
overrides the reference's defaults.  Operators of the reference outside the path
(load balancing, snapshots, restarts, analysis, ghost exchanges -- one GPU holds
the whole periodic box, images are resolved inside the library) are accepted as
no-ops; any other operator name raises ``DeckError``, as exaStamp fails on an
unknown operator.

The particle-update graph of config_move_particles.msp (trigger_move_particles,
update_particles_full/fast, parallel_update_particles, update_particle_neighbors) is
restated node for node, with particle_displ_over (and its async form of
config_speculative_verlet.msp) as the trigger and chunk_neighbors as the list
build, so decks that override any of these nodes run as written.

Differences that a deck cannot see in its results: the Newton-symmetric variants
(``eam_symmetry: true``, ``lj_compute_force_symetric``) evaluate each pair from both
of its atoms, with a pair scalar symmetric in them; ``chunk_size`` is accepted
and does not change the list; the random streams of ``gaussian_noise_r/v`` are
numpy Philox streams (seed ``--seed``), not exaNBody's.

    python -m exastamp_amd.deck single_specy_nosym.msp --set-global-max_iteration 20
"""
from __future__ import annotations

import argparse
import copy
import dataclasses
import math
import sys
from pathlib import Path

import numpy as np
import yaml

from .inputs import Config
from .units import AMU_KG, EV, KB, PRESSURE_UNIT_PA, parse_quantity

AMU_G = AMU_KG * 1e3


class DeckError(RuntimeError):
    """A deck the runner cannot execute (unknown operator, bad slot value)."""


# Default graph: the reference's node names and control flow for the NVE path.
DEFAULT_GRAPH = """
global:
  max_iteration: 1000
  timestep: 0
  physical_time: 0.
  dt: 1.0e-3 ps
  rcut_inc: 1.0 ang
  simulation_thermostate_screen_frequency: 10
  simulation_thermostate_file_frequency: 10
  log_mode: mechanical
  thermostate_file: "thermodynamic_state.csv"
  trigger_thermo_state: true
  md_loop_continue: true
init_parameters: nop
generate_default_species: species
compute_force_prolog: zero_force_energy
compute_force: nop
compute_force_epilog: force_to_accel
compute_all_forces_energy:
  - compute_force_prolog
  - compute_force
  - compute_force_epilog
verlet_first_half:
  - push_f_v_r: { dt_scale: 1.0, xform_mode: INV_XFORM }
  - push_f_v: { dt_scale: 0.5, xform_mode: IDENTITY }
verlet_second_half:
  - push_f_v: { dt_scale: 0.5, xform_mode: IDENTITY }
numerical_scheme: verlet_nve
verlet_nve:
  name: NVE_scheme
  body:
    - verlet_first_half
    - check_and_update_particles
    - compute_all_forces_energy
    - verlet_second_half
chunk_neighbors:
  config:
    chunk_size: 1
chunk_neighbors_impl: chunk_neighbors
update_particle_neighbors:
  - amr_grid_pairs
  - chunk_neighbors_impl
  - resize_particle_locks
parallel_update_particles:
  - migrate_cell_particles
  - rebuild_amr
  - backup_r
  - ghost_full_update
  - grid_post_processing
  - update_particle_neighbors
update_particles_full_body:
  - move_particles
  - trigger_load_balance
  - load_balancing_if_triggered
  - parallel_update_particles
update_particles_full:
  condition: trigger_move_particles
  body:
    - update_particles_full_body
update_particles_fast_body:
  - ghost_update_r
update_particles_fast:
  condition: not trigger_move_particles
  body:
    - update_particles_fast_body
trigger_move_particles:
  rebind: { threshold: max_displ , result: trigger_move_particles }
  body:
    - particle_displ_over
check_and_update_particles:
  - trigger_move_particles
  - update_particles_full
  - update_particles_fast
  - loadbalance_log_helper:
      rebind: { lb_flag: trigger_load_balance , move_flag: trigger_move_particles }
      body: [ lb_event_counter ]
begin_iteration:
  - trigger_thermostate_screen
  - trigger_thermostate_file
end_iteration:
  - thermostate_compute_if_triggered
  - thermostate_screen_if_triggered
  - thermostate_file_if_triggered
first_iteration:
  - init_particles
  - compute_all_forces_energy
  - default_thermostate_compute
  - default_thermostate_screen: { lb_flag: false , move_flag: false , print_header: true }
  - default_thermostate_file
  - next_time_step
md_trajectory_loop:
  loop: true
  name: md_loop
  condition: md_loop_continue
  body:
    - begin_iteration
    - numerical_scheme
    - end_iteration
    - next_time_step
    - md_loop_stop
md_loop_stop:
  rebind: { end_at: max_iteration , result: md_loop_continue }
  body:
    - sim_continue
simulation_epilog: nop
simulation:
  name: exaStamp_simulation
  body:
    - global
    - init_parameters
    - generate_default_species
    - setup_system
    - init_rcut_max
    - first_iteration
    - md_trajectory_loop
    - simulation_epilog
"""

# Operators of the reference that have nothing to do on one GPU or outside the path.
NOOPS = {
    "nop", "print_logo_banner", "print_version_info", "message", "hw_device_init", "hw_device_finalize",
    "mpi_comm_world", "init_cuda", "finalize_cuda", "update_ghost_config", "make_empty_grid", "grid_flavor",
    "grid_flavor_full", "grid_flavor_multimat", "grid_flavor_minimal", "particle_regions", "init_prolog",
    "init_epilog", "init_rcb_grid", "grid_post_processing",
    "reduce_species_after_read", "print_domain", "performance_adviser", "memory_stats", "grid_stats",
    "load_balance_auto_tune_start", "load_balance_auto_tune_end", "nose_hoover_additional_step",
    "md_loop_prolog", "md_loop_epilog", "trigger_restart", "trigger_analysis", "trigger_snapshot",
    "write_restart_if_triggered", "perform_analysis_if_triggered", "write_snapshot_if_triggered",
    "write_final_restart", "write_restart", "ghost_update_r", "ghost_update_opt", "ghost_update_all_no_fv",
    "update_force_energy_from_ghost", "ghost_config", "ghost_config_opt", "configuration", "preinit_rcut_max",
    "xxx_simulation_epilog",
    # particle moves on one GPU: migration, load balancing, AMR sub-cells, ghost layers and
    # position backups have nothing to do (the list build keeps the reference positions)
    "move_particles", "extend_domain", "load_balance", "trigger_load_balance", "load_balancing_if_triggered",
    "migrate_cell_particles", "rebuild_amr", "backup_r", "ghost_full_update", "ghost_comm_scheme",
    "profile_ghost_comm_scheme", "ghost_update_all_impl", "grid_memory_compact", "amr_grid_pairs",
    "resize_particle_locks", "compute_primary_neighbors", "compute_dual_neighbors", "lb_event_counter",
    # a consistency check of exaNBody's chunk streams; the lists here are checked by the tests
    "verify_chunk_neighbors",
    "ghost_update_emb", "update_opt_from_ghost", "update_rho_from_ghost",
}


def _merge(base, over):
    """Deck override: maps merge recursively, anything else replaces; '+key' appends."""
    if not isinstance(base, dict) or not isinstance(over, dict):
        return copy.deepcopy(over)
    out = dict(base)
    for k, v in over.items():
        if isinstance(k, str) and k.startswith("+"):
            key = k[1:]
            prev = out.get(key) or []
            out[key] = list(prev if isinstance(prev, list) else [prev]) + list(v if isinstance(v, list) else [v])
        elif k in out:
            out[k] = _merge(out[k], v)
        else:
            out[k] = copy.deepcopy(v)
    return out


def _read_yaml(path: Path) -> dict:
    with open(path) as f:
        doc = yaml.safe_load(f)
    if doc is None:
        return {}
    if not isinstance(doc, dict):
        raise DeckError(f"{path}: a deck is a map of node definitions")
    return doc


def load_deck(path, search=(), sets=()) -> dict:
    """The deck at `path` merged over the default graph, includes resolved (relative
    to the including file, then the directories in `search`), then `sets`
    overrides applied: (["global", "max_iteration"], "20") pairs."""
    path = Path(path)
    seen = []

    def load(p: Path) -> dict:
        p = p.resolve()
        if p in seen:
            raise DeckError(f"include cycle through {p}")
        seen.append(p)
        doc = _read_yaml(p)
        merged = {}
        for inc in doc.pop("includes", None) or []:
            q = _find(str(inc), p.parent, search)
            merged = _merge(merged, load(q))
        seen.pop()
        return _merge(merged, doc)

    cfg = _merge(yaml.safe_load(DEFAULT_GRAPH), load(path))
    for keys, value in sets:
        node = cfg
        for k in keys[:-1]:
            node = node.setdefault(k, {})
            if not isinstance(node, dict):
                raise DeckError(f"--set-{'-'.join(keys)}: {k} is not a map")
        node[keys[-1]] = yaml.safe_load(value)
    cfg["__deck_dir__"] = str(path.resolve().parent)
    cfg["__search__"] = [str(s) for s in search]
    return cfg


def _find(name: str, here: Path, search) -> Path:
    for d in [here, *[Path(s) for s in search]]:
        if (d / name).exists():
            return d / name
    raise DeckError(f"cannot find {name!r} (looked in {here} and {list(map(str, search))})")


# --- lattices (exaNBody's lattice operator; bulk_lattice.cpp:17-31 wraps it) -------
_BASES = {
    "SC": np.zeros((1, 3)),
    "BCC": np.array([[0.0, 0.0, 0.0], [0.5, 0.5, 0.5]]),
    "FCC": np.array([[0.0, 0.0, 0.0], [0.5, 0.5, 0.0], [0.5, 0.0, 0.5], [0.0, 0.5, 0.5]]),
}


def _quantity_list(v):
    return [parse_quantity(x) for x in v]


@dataclasses.dataclass
class ThermoRecord:
    """One thermodynamic state with the quantities and conversions of the reference's
    outputs (print_thermodynamic_state.cpp:223-282, dump_thermodynamic_state.cpp:84-122):
    energies per particle in eV, temperatures in K, pressures in Pa, box lengths and
    volume in A and A^3, density in g/cm^3.  p_full holds the full stress tensor
    (virial + kinetic tensor) / V in the order xx yy zz xy xz yz, p_vir the virial
    part / V of xx yy zz."""
    step: int
    time_ps: float
    particles: int
    total_ev: float      # per particle
    kinetic_ev: float
    potential_ev: float
    temperature_k: float
    t_xyz: tuple         # Tx Ty Tz
    pressure_pa: float   # hydrostatic, (kinetic + virial) trace / 3V
    p_full: tuple        # full stress tensor xx yy zz xy xz yz
    p_vir: tuple         # virial stress xx yy zz
    vonmises_pa: float
    lengths: tuple       # A B C
    volume: float
    mass: float          # Da
    density: float       # g/cm^3
    angles: tuple = (90.0, 90.0, 90.0)  # alpha beta gamma, degrees

    def line(self) -> str:
        """The row dump_thermodynamic_state writes (dump_thermodynamic_state.cpp:101-121),
        without the newline."""
        return CSV_ROW % (self.step, self.time_ps, self.particles, self.total_ev, self.kinetic_ev,
                          self.potential_ev, self.temperature_k, *self.p_full, *self.lengths, *self.angles,
                          self.volume, self.density)

    def log_values(self) -> dict:
        """Values of the screen log items (print_thermodynamic_state.cpp:254-282)."""
        return {"stp": float(self.step), "pht": self.time_ps, "prt": float(self.particles), "sta": 0.0,
                "toe": self.total_ev, "kie": self.kinetic_ev, "poe": self.potential_ev, "ele": 0.0,
                "tmp": self.temperature_k, "tmx": self.t_xyz[0], "tmy": self.t_xyz[1], "tmz": self.t_xyz[2],
                "pre": self.pressure_pa, "prx": self.p_vir[0], "pry": self.p_vir[1], "prz": self.p_vir[2],
                "pxy": self.p_full[3], "pxz": self.p_full[4], "pyz": self.p_full[5], "smi": self.vonmises_pa,
                "vol": self.volume, "mas": self.mass, "bxa": self.lengths[0], "bxb": self.lengths[1],
                "bxc": self.lengths[2], "baa": self.angles[0], "bab": self.angles[1], "bag": self.angles[2],
                "rho": self.density}


def cell_geometry(xform, extent):
    """Box edge lengths A, B, C and angles alpha, beta, gamma (degrees) of the domain
    as print_thermodynamic_state.cpp:252-262 and dump_thermodynamic_state.cpp:90-99
    compute them: a, b, c = xform times the grid box edges; the three angles all divide
    by B*C there, which this keeps so the outputs agree (it only matters for a
    non-orthogonal xform with B*C != C*A or A*B)."""
    m = np.asarray(xform, dtype=np.float64)
    e = np.asarray(extent, dtype=np.float64)
    a, b, c = m[:, 0] * e[0], m[:, 1] * e[1], m[:, 2] * e[2]
    A, B, C = (float(math.sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2])) for v in (a, b, c))

    def dot(u, w):
        return float(u[0] * w[0] + u[1] * w[1] + u[2] * w[2])

    def ang(x):
        return math.acos(x) / math.acos(-1.0) * 180.0 if -1.0 <= x <= 1.0 else float("nan")

    if B * C == 0.0:
        return (A, B, C), (90.0, 90.0, 90.0)
    return (A, B, C), (ang(dot(b, c) / (B * C)), ang(dot(c, a) / (B * C)), ang(dot(a, b) / (B * C)))


# the file row and header of dump_thermodynamic_state (dump_thermodynamic_state.cpp:61,101)
CSV_ROW = ("%9d % .6e %13d  % .10e  % .10e  % .10e  % 9.12f  % 9.12f  % 9.12f  % 9.12f  % 9.12f  % 9.12f "
           "% 9.12f % 12.12f % 12.12f % 12.12f % 9.12f % 9.12f % 9.12f % 16.12f % 13.12f ")
THERMO_HEADER = ("# Step     Time (ps)     Particles  Tot. E. (eV/part)  Kin. E. (eV/part)  Pot. E. (eV/part)  "
                 "Temp. (K) Pxx Pyy Pzz Pxy Pxz Pyz (Pa) A/B/C (ang)    alpha/beta/gamma (deg)     Vol. (ang^3)  "
                 "Rho (g/cm^3)")

# Screen log items of print_thermodynamic_state: key -> (header, printf format)
# (thermodynamic_log_config.h:136-165), and the item lists of its log modes
# (print_thermodynamic_state.cpp:63-201).  A mode it does not know keeps the
# default item list (its keyword-list parser adds no items).
LOG_ITEMS = {
    "stp": ("Step", "% 9.0f"), "pht": ("Time (ps)", "% .6e"), "prt": ("Particles", "% 12.0f"),
    "sta": ("Mv/Ext/Imb.", "%.1e"), "toe": ("Tot. E. (eV/part)", "% .10e"),
    "kie": ("Kin. E. (eV/part)", "% .10e"), "poe": ("Pot. E. (eV/part)", "% .10e"),
    "ele": ("Elec. E. (eV/part)", "% .10e"), "tmp": ("Temp. (K)", "% 10.3f"), "tmx": ("   Tx (K)", "% 10.3f"),
    "tmy": ("   Ty (K)", "% 10.3f"), "tmz": ("   Tz (K)", "% 10.3f"), "pre": ("Press. (Pa)", "% 11.3e"),
    "prx": ("    Px (Pa)", "% 11.3e"), "pry": ("    Py (Pa)", "% 11.3e"), "prz": ("    Pz (Pa)", "% 11.3e"),
    "pxy": ("   Pxy (Pa)", "% 11.3e"), "pxz": ("   Pxz (Pa)", "% 11.3e"), "pyz": ("   Pyz (Pa)", "% 11.3e"),
    "smi": ("sMises (Pa)", "% .3e"), "vol": ("Vol. (ang^3)", "% 13.6e"), "mas": ("Mass", "% .3e"),
    "bxa": ("A (ang)", "% .3f"), "bxb": ("B (ang)", "% .3f"), "bxc": ("C (ang)", "% .3f"),
    "baa": ("alpha (deg)", "% 12.3f"), "bab": ("beta (deg)", "% 12.3f"), "bag": ("gamma (deg)", "% 12.3f"),
    "rho": ("Rho (g/cm^3)", "% 12.6f"),
}
_BASIC = ["stp", "pht", "toe", "kie", "poe", "tmp", "pre"]
_FULL = ["stp", "pht", "toe", "kie", "poe", "tmp", "tmx", "tmy", "tmz", "pre", "prx", "pry", "prz"]
LOG_MODES = {
    "default": _BASIC + ["sta"], "thermo_basic": _BASIC + ["sta"],
    "thermo": _FULL + ["sta"], "thermo_full": _FULL + ["sta"],
    "vol_fluct_ortho_basic": _BASIC + ["vol", "bxa", "bxb", "bxc", "rho", "sta"],
    "vol_fluct_ortho": _FULL + ["vol", "bxa", "bxb", "bxc", "rho", "sta"],
    "vol_fluct_ortho_full": _FULL + ["vol", "bxa", "bxb", "bxc", "rho", "sta"],
    "vol_fluct_tricl_basic": _BASIC + ["vol", "bxa", "bxb", "bxc", "baa", "bab", "bag", "rho", "sta"],
    "vol_fluct_tricl": _FULL + ["pxy", "pxz", "pyz", "vol", "bxa", "bxb", "bxc", "baa", "bab", "bag", "rho", "sta"],
    "vol_fluct_tricl_full": _FULL + ["pxy", "pxz", "pyz", "vol", "bxa", "bxb", "bxc", "baa", "bab", "bag", "rho",
                                     "sta"],
    "mechanical": ["stp", "pht", "prt", "sta", "toe", "kie", "poe", "tmp", "pre", "smi", "vol", "mas"],
}
LOG_DEFAULT_ITEMS = ["stp", "pht", "prt", "sta", "toe", "kie", "poe", "tmp", "pre", "vol"]


def _log_width(key: str) -> int:
    header, fmt = LOG_ITEMS[key]
    return max(len(fmt % 0.0) + (3 if key == "sta" else 0), len(header))


def log_header(mode: str) -> str:
    """The header line print_thermodynamic_state prints (thermodynamic_log_config.h:86-90)."""
    return "".join(" %*s" % (_log_width(k), LOG_ITEMS[k][0]) for k in LOG_MODES.get(mode, LOG_DEFAULT_ITEMS))


def _moves_char(count: int, one: str, many: str) -> str:
    if count <= 0:
        return " "
    return one if count == 1 else (str(count) if count < 10 else many)


def log_line(rec: ThermoRecord, mode: str, moves: int = 0) -> str:
    """One screen line (thermodynamic_log_config.h:91-127): the status column shows the
    particle moves (list rebuilds) since the last line; there is no load balancing
    and no domain extension on one GPU."""
    vals = rec.log_values()
    out = []
    for k in LOG_MODES.get(mode, LOG_DEFAULT_ITEMS):
        if k == "sta":
            out.append(" %c %c%*s" % (_moves_char(moves, "m", "M"), " ", _log_width(k) - 3, ""))
        else:
            out.append(" " + LOG_ITEMS[k][1] % vals[k])
    return "".join(out)


G_PER_CM3_PER_DA_PER_A3 = AMU_G * 1e24


class Runner:
    """Executes a loaded deck on one GPU through the operator mirror."""

    def __init__(self, cfg: dict, device: int = 0, mixed: bool = False, seed: int = 0, out=None,
                 thermo_file: str | None = None):
        from .operators import Simulation  # the C ABI is loaded only when a deck runs
        self.cfg = cfg
        self.mixed = mixed
        self.seed = seed
        self.out = out if out is not None else sys.stdout
        self.thermo_file = thermo_file
        self.sim = Simulation(device)
        self.slots: dict = {"rcut_max": 0.0}
        self.rebind: list[dict] = []
        self.records: list[ThermoRecord] = []
        self.species: list[tuple[str, float]] = []
        self.type_map: dict[str, int] = {}
        self.domain: dict = {}
        self.atoms: Config | None = None
        self.init_atoms: Config | None = None  # the configuration the MD started from
        self.tables_loaded = None
        self.dry = False
        self._file = None
        self.rebuilds = 0
        self.rebuilds_printed = 0
        self.displ_pending = None

    # --- slots with rebind ----------------------------------------------------
    def _slot_name(self, name):
        for m in reversed(self.rebind):
            if name in m:
                return m[name]
        return name

    def get(self, name, default=None):
        return self.slots.get(self._slot_name(name), default)

    def set(self, name, value):
        self.slots[self._slot_name(name)] = value

    # --- graph execution ------------------------------------------------------
    def run(self) -> list[ThermoRecord]:
        try:
            self.node("simulation")
        finally:
            if self._file:
                self._file.close()
        return self.records

    def node(self, name: str, params=None):
        ops = _OPS
        d = self.cfg.get(name, None) if name in self.cfg else _MISSING
        if isinstance(d, str):
            return self.node(d, params)
        if isinstance(d, list) and name in ops:  # an operator given a list value (species: [...])
            return ops[name](self, _merge({"value": d}, params or {}))
        if isinstance(d, list):
            if params:
                raise DeckError(f"{name} is a batch; it takes no parameters")
            for item in d:
                self.item(item)
            return None
        if isinstance(d, dict) and "body" in d:
            return self.block(name, d)
        own = d if isinstance(d, dict) else {}
        p = _merge(own, params or {})
        if name in ops:
            return ops[name](self, p)
        if name in NOOPS:
            return None
        raise DeckError(f"unknown operator {name!r}")

    def item(self, item):
        if isinstance(item, str):
            return self.node(item)
        if isinstance(item, dict) and len(item) == 1:
            (k, v), = item.items()
            if isinstance(v, dict) and "body" in v:  # a block defined in place
                return self.block(k, v)
            return self.node(k, v if isinstance(v, dict) else ({} if v is None else {"value": v}))
        raise DeckError(f"cannot read batch item {item!r}")

    def block(self, name, d):
        self.rebind.append(dict(d.get("rebind") or {}))
        try:
            body = d.get("body") or []
            if d.get("loop"):
                cond = d.get("condition")
                if cond is None:
                    raise DeckError(f"loop {name} has no condition")
                while self.condition(cond):
                    for item in body:
                        self.item(item)
            else:
                if d.get("condition") is not None and not self.condition(d["condition"]):
                    return None
                for item in body:
                    self.item(item)
        finally:
            self.rebind.pop()
        return None

    def condition(self, cond) -> bool:
        """A block condition: a slot name, or "not" and a slot name."""
        if isinstance(cond, bool):
            return cond
        words = str(cond).split()
        if len(words) == 2 and words[0] == "not":
            return not bool(self.get(words[1], False))
        return bool(self.get(str(cond), True))

    # --- helpers ----------------------------------------------------------------
    def path(self, name: str) -> Path:
        return _find(name, Path(self.cfg["__deck_dir__"]), self.cfg.get("__search__", []))

    def dt(self) -> float:
        return parse_quantity(self.get("dt"))

    def thermo(self) -> ThermoRecord:
        st = self.sim.simulation_thermodynamic_state()
        n = st.particle_count
        v = st.volume
        kt = 2.0 * (st.kinetic_tensor - 0.5 * np.outer(st.momentum, st.momentum) / st.mass)
        vir = st.virial
        full = (vir + kt) / v * PRESSURE_UNIT_PA
        ke = st.raw[21:24] - 0.5 * st.momentum ** 2 / st.mass
        d, o = np.diag(vir), (vir[0, 1], vir[0, 2], vir[1, 2])
        mises = np.sqrt(0.5 * ((d[0] - d[1]) ** 2 + (d[1] - d[2]) ** 2 + (d[2] - d[0]) ** 2
                               + 6.0 * (o[0] ** 2 + o[1] ** 2 + o[2] ** 2))) / v
        a = self.atoms
        lengths, angles = cell_geometry(self.sim.xform, a.hi[0] - a.lo[0] if a is not None else np.zeros(3))
        rec = ThermoRecord(step=int(self.get("timestep", 0)), time_ps=float(self.get("physical_time", 0.0)),
                           particles=n, total_ev=st.total_energy / EV / n, kinetic_ev=st.kinetic_energy / EV / n,
                           potential_ev=st.potential_energy / EV / n, temperature_k=st.temperature,
                           t_xyz=tuple(float(2.0 * x / (n * KB)) for x in ke),
                           pressure_pa=st.pressure_pa,
                           p_full=tuple(float(full[i, j]) for i, j in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))),
                           p_vir=tuple(float(vir[k, k] / v * PRESSURE_UNIT_PA) for k in range(3)),
                           vonmises_pa=float(mises * PRESSURE_UNIT_PA), lengths=lengths, volume=v, mass=st.mass,
                           density=st.mass / v * G_PER_CM3_PER_DA_PER_A3, angles=angles)
        self.records.append(rec)
        return rec


_MISSING = object()


def _op_global(r: Runner, p):
    for k, v in p.items():
        r.set(k, v)


def _op_species(r: Runner, p):
    spec = p.get("species", p.get("value"))
    if spec is None and p and "verbose" not in p and "fail_if_empty" not in p:
        spec = p
    if not spec:
        if p.get("fail_if_empty") and not r.species:
            raise DeckError("no species defined")
        return
    out = []
    for s in spec if isinstance(spec, list) else [spec]:
        for name, props in s.items():
            out.append((name, parse_quantity(props["mass"])))
    r.species = out


def _op_particle_types(r: Runner, p):
    r.type_map = {k: int(v) for k, v in (p.get("particle_type_map") or {}).items()}


def _op_particle_type_add_properties(r: Runner, p):
    masses = {}
    for name, props in p.items():
        if isinstance(props, dict) and "mass" in props:
            masses[name] = parse_quantity(props["mass"])
    if not r.type_map:
        r.type_map = {n: i for i, n in enumerate(masses)}
    spec = sorted(r.type_map.items(), key=lambda kv: kv[1])
    known = dict(r.species)
    r.species = [(n, masses.get(n, known.get(n))) for n, _ in spec]
    if any(m is None for _, m in r.species):
        raise DeckError("particle_type_add_properties: a type has no mass")


def _op_domain(r: Runner, p):
    d = dict(r.domain)
    d.update(p)
    xf = d.get("xform")
    if xf is not None:
        m = np.asarray(xf, dtype=float)
        if m.shape != (3, 3) or not np.all(np.isfinite(m)) or not np.linalg.det(m) > 0.0:
            raise DeckError("domain: xform must be a 3x3 matrix with a positive determinant")
    r.domain = d


def _op_lattice(r: Runner, p):
    struct = str(p.get("structure", "FCC")).upper()
    if struct not in _BASES:
        raise DeckError(f"lattice: structure {struct} is not supported (SC, BCC, FCC)")
    basis = _BASES[struct]
    types = p.get("types") or []
    if len(types) != len(basis):
        raise DeckError(f"lattice: {struct} needs {len(basis)} types, got {len(types)}")
    size = np.asarray(_quantity_list(p["size"]))
    b = r.domain.get("bounds")
    if b is None:
        raise DeckError("lattice: the domain has no bounds")
    lo = np.asarray(_quantity_list(b[0]))
    hi = np.asarray(_quantity_list(b[1]))
    reps = np.rint((hi - lo) / size).astype(int)
    if np.any(reps < 1) or not np.allclose(reps * size, hi - lo, rtol=1e-9, atol=1e-9):
        raise DeckError("lattice: the domain is not a whole number of unit cells")
    ii, jj, kk = np.meshgrid(np.arange(reps[0]), np.arange(reps[1]), np.arange(reps[2]), indexing="ij")
    cells = np.stack([ii.ravel(), jj.ravel(), kk.ravel()], axis=1).astype(float)
    pos = (cells[:, None, :] + basis[None, :, :]).reshape(-1, 3) * size + lo
    tmap = r.type_map or {n: i for i, (n, _) in enumerate(r.species)}
    tb = np.asarray([tmap[t] for t in types], dtype=np.uint8)
    typ = np.tile(tb, cells.shape[0])
    per = tuple(int(bool(x)) for x in r.domain.get("periodic", [True, True, True]))
    r.atoms = Config(r=pos, v=np.zeros_like(pos), type=typ, lo=lo[None, :], hi=hi[None, :], periodic=per)


def _op_gaussian_noise_r(r: Runner, p):
    if r.atoms is None:
        raise DeckError("gaussian_noise_r before any atoms")
    sigma = parse_quantity(p.get("sigma", 0.0))
    g = np.random.Generator(np.random.Philox(key=r.seed * 2 + 0))
    a = r.atoms
    a.r = a.r + g.normal(scale=sigma, size=a.r.shape)
    lo, hi = a.lo[0], a.hi[0]
    for k in range(3):  # wrap along periodic axes, as the grid does on insertion
        if a.periodic[k]:
            a.r[:, k] = lo[k] + np.mod(a.r[:, k] - lo[k], hi[k] - lo[k])


def _op_gaussian_noise_v(r: Runner, p):
    if r.atoms is None:
        raise DeckError("gaussian_noise_v before any atoms")
    sigma = parse_quantity(p.get("sigma", 0.0))
    g = np.random.Generator(np.random.Philox(key=r.seed * 2 + 1))
    r.atoms.v = r.atoms.v + g.normal(scale=sigma, size=r.atoms.v.shape)


def _op_setup_species_check(r: Runner):
    if not r.species:
        raise DeckError("no species defined")


def _op_init_rcut_max(r: Runner, p):
    # executing the force nodes on an empty system only publishes their rcut
    r.dry = True
    try:
        r.node("compute_force")
    finally:
        r.dry = False
    _op_nbh_dist(r, {})


def _op_init_particles(r: Runner, p):
    if r.atoms is None:
        raise DeckError("init_particles: setup_system produced no atoms")
    _op_setup_species_check(r)
    r.sim.species(r.species)
    r.sim.set_config(r.atoms)
    xf = r.domain.get("xform")
    if xf is not None and not np.array_equal(np.asarray(xf, dtype=float), np.eye(3)):
        r.sim.set_xform(np.asarray(xf, dtype=float))
    r.init_atoms = copy.deepcopy(r.atoms)
    if r.tables_loaded is not None:
        r.sim.eam_alloy_init(r.tables_loaded)
    r.node("update_particle_neighbors")


def _build_list(r: Runner):
    rmax = float(r.get("rcut_max", 0.0))
    if rmax <= 0.0:
        raise DeckError("no force operator published rcut_max (compute_force is empty?)")
    conf = (r.cfg.get("chunk_neighbors") or {}).get("config") or {}
    r.sim.chunk_neighbors(rcut_max=rmax, rcut_inc=parse_quantity(r.get("rcut_inc")), config=conf)
    r.rebuilds += 1


def _op_chunk_neighbors(r: Runner, p):
    _build_list(r)


def _op_nbh_dist(r: Runner, p):
    # the move tolerance: max_displ = rcut_inc / 2 (config_move_particles.msp:116-118)
    r.set("max_displ", 0.5 * parse_quantity(r.get("rcut_inc")))


def _op_particle_displ_over(r: Runner, p):
    """particle_displ_over: result = some atom moved more than threshold since the last
    list build; with async: true the result is published by particle_displ_over_async_end."""
    th = r.get("threshold", None)
    if th is None:
        th = 0.5 * parse_quantity(r.get("rcut_inc"))
    over = r.sim.particle_displ_over(parse_quantity(th))
    if p.get("async", False):
        r.displ_pending = over
    else:
        r.set("result", over)


def _op_particle_displ_over_async_end(r: Runner, p):
    if r.displ_pending is None:
        raise DeckError("particle_displ_over_async_end without a started particle_displ_over")
    r.set("result", r.displ_pending)
    r.displ_pending = None


def _publish_rcut(r: Runner, rc):
    r.set("rcut_max", max(float(r.get("rcut_max", 0.0) or 0.0), rc))


def _trigger(r: Runner) -> bool:
    return bool(r.get("trigger_thermo_state", False))


def _op_lj(r: Runner, p, symmetric=False):
    rc = parse_quantity(p["rcut"])
    _publish_rcut(r, rc)
    if r.dry:
        return
    r.sim.lj_compute_force(parameters=p["parameters"], rcut=rc, trigger_thermo_state=_trigger(r),
                           compute_virial=bool(p.get("compute_virial", True)), mixed=r.mixed,
                           symmetric=symmetric, type=p.get("type"))


def _op_lj_symetric(r: Runner, p):
    _op_lj(r, p, symmetric=True)


def _lj_energy(eps, sigma, rr):
    # lj_compute_energy (lennard_jones.h:40-50)
    ratio = sigma / rr
    r6 = ratio ** 6
    r12 = r6 * r6
    return 4.0 * eps * (r12 - r6), (-24.0 * eps * (2.0 * r12 - r6)) / rr


def _op_lj_plot(r: Runner, p):
    """lj_plot (pair_potential_plot.cpp:45-103): e(r), de/dr and their central-difference
    check at r = i rcut / samples (0 < i < samples), one line each, in `file`
    (default lj.csv), values in internal units, C++ stream formatting."""
    eps = parse_quantity(p["parameters"]["epsilon"])
    sig = parse_quantity(p["parameters"]["sigma"])
    rc = parse_quantity(p["rcut"])
    n = int(p.get("samples", 1000))
    step = rc / n
    small = step * 1.0e-2
    with open(str(p.get("file", "lj.csv")), "w") as out:
        for i in range(1, n):
            rr = i * step
            e1, _ = _lj_energy(eps, sig, rr - small)
            e2, _ = _lj_energy(eps, sig, rr + small)
            e, de = _lj_energy(eps, sig, rr)
            approx = (e2 - e1) / (2.0 * small)
            diff = approx - de
            ampl = max(abs(approx), abs(de))
            if ampl > 0.0:
                diff /= ampl
            out.write(" ".join(format(x, "g") for x in (rr, e, de, approx, diff)) + "\n")


def _op_lj_multi(r: Runner, p):
    rc = parse_quantity(p["rcut"])
    pairs = p.get("parameters") or []
    _publish_rcut(r, max([rc] + [parse_quantity(e["rcut"]) for e in pairs]))
    if r.dry:
        return
    r.sim.lj_multi_force(rcut=rc, parameters=pairs, common_parameters=p.get("common_parameters"),
                         trigger_thermo_state=_trigger(r), compute_virial=bool(p.get("compute_virial", True)),
                         mixed=r.mixed)


def _tables_from(r: Runner, params):
    f = params.get("file") if isinstance(params, dict) else None
    if f is None:
        raise DeckError("eam_alloy parameters need a file")
    from .potentials import read_setfl
    return read_setfl(r.path(str(f)))


def _op_eam_alloy_init(r: Runner, p):
    t = _tables_from(r, p.get("parameters") or {})
    r.set("parameters", t)
    r.tables_loaded = t


def _op_eam_alloy_force(r: Runner, p):
    rc = parse_quantity(p["rcut"])
    _publish_rcut(r, rc)
    if p.get("parameters") is not None and isinstance(p["parameters"], dict) and r.tables_loaded is None:
        r.tables_loaded = _tables_from(r, p["parameters"])   # single-pass decks give the file inline
        if r.atoms is not None and r.sim.n:
            r.sim.eam_alloy_init(r.tables_loaded)
    if r.dry:
        return
    if r.tables_loaded is None:
        raise DeckError("eam_alloy_force: no tables (eam_alloy_init did not run)")
    flag = lambda k: bool(p.get(k, True))
    r.sim.eam_alloy_force(rcut=rc, eam_rho=flag("eam_rho"), eam_rho2emb=flag("eam_rho2emb"),
                          eam_ghost=flag("eam_ghost"), eam_force=flag("eam_force"),
                          eam_symmetry=bool(p.get("eam_symmetry", False)), trigger_thermo_state=_trigger(r),
                          compute_virial=bool(p.get("compute_virial", False)), mixed=r.mixed,
                          types=p.get("types") or None)


def _op_johnson_init(r: Runner, p):
    """johnson_init (eam_potential.cu:62-70): its `parameters` slot is an OUTPUT, read by
    the Johnson force operators through the shared slot."""
    if p.get("parameters") is None:
        raise DeckError("johnson_init: parameters missing")
    r.set("parameters", p["parameters"])


def _op_johnson(r: Runner, p, op="johnson_force"):
    rc = parse_quantity(p["rcut"])
    _publish_rcut(r, rc)
    params = p.get("parameters")
    if params is None:
        params = r.get("parameters")   # set by johnson_init (INPUT_OUTPUT slot, eam_potential.cu:92)
    if not isinstance(params, dict):
        raise DeckError(f"{op}: no parameters (give them to the operator or run johnson_init first)")
    if r.dry:
        return
    kw = {} if op == "johnson_emb" else {"compute_virial": bool(p.get("compute_virial", False))}
    getattr(r.sim, op)(rcut=rc, parameters=params, **kw)


def _op_zero(r: Runner, p):
    if not r.dry:
        r.sim.zero_force_energy()


def _op_accel(r: Runner, p):
    if not r.dry:
        r.sim.force_to_accel()


def _op_push_f_v_r(r: Runner, p):
    r.sim.push_f_v_r(r.dt(), dt_scale=float(p.get("dt_scale", 1.0)), xform_mode=p.get("xform_mode", "INV_XFORM"))


def _op_push_f_v(r: Runner, p):
    r.sim.push_f_v(r.dt(), dt_scale=float(p.get("dt_scale", 0.5)), xform_mode=p.get("xform_mode", "IDENTITY"))


def _freq_hit(r: Runner, key) -> bool:
    f = int(r.get(key, -1) or -1)
    step = int(r.get("timestep", 0))
    last = step >= int(r.get("max_iteration", 0))
    return f > 0 and (step % f == 0 or last)


def _op_trigger_screen(r: Runner, p):
    r.set("trigger_thermo_screen", _freq_hit(r, "simulation_thermostate_screen_frequency"))
    r.set("trigger_thermo_state", bool(r.get("trigger_thermo_screen")) or bool(r.get("trigger_thermo_file")))


def _op_trigger_file(r: Runner, p):
    r.set("trigger_thermo_file", _freq_hit(r, "simulation_thermostate_file_frequency"))
    r.set("trigger_thermo_state", bool(r.get("trigger_thermo_screen")) or bool(r.get("trigger_thermo_file")))


def _op_thermo_compute_if(r: Runner, p):
    if _trigger(r):
        r.thermo()


def _screen(r: Runner, header: bool):
    mode = str(r.get("log_mode", "default"))
    if header:
        print(log_header(mode), file=r.out)
    print(log_line(r.records[-1], mode, r.rebuilds - r.rebuilds_printed), file=r.out)
    r.rebuilds_printed = r.rebuilds


def _op_thermo_screen_if(r: Runner, p):
    if r.get("trigger_thermo_screen") and r.records and r.records[-1].step == int(r.get("timestep", 0)):
        _screen(r, bool(p.get("print_header", False)))


def _op_thermo_file_if(r: Runner, p):
    if r.get("trigger_thermo_file") and r.records and r.records[-1].step == int(r.get("timestep", 0)):
        _write_file(r, r.records[-1])


def _write_file(r: Runner, rec: ThermoRecord):
    name = r.thermo_file
    if name is None:
        return
    if r._file is None:
        r._file = open(name, "w")
        print(THERMO_HEADER, file=r._file)
    print(rec.line(), file=r._file)


def _op_default_thermo_compute(r: Runner, p):
    r.thermo()


def _op_default_thermo_screen(r: Runner, p):
    _screen(r, bool(p.get("print_header", False)))


def _op_default_thermo_file(r: Runner, p):
    if int(r.get("simulation_thermostate_file_frequency", -1) or -1) > 0:
        _write_file(r, r.records[-1])


def _op_next_time_step(r: Runner, p):
    r.set("timestep", int(r.get("timestep", 0)) + 1)
    r.set("physical_time", float(r.get("physical_time", 0.0)) + r.dt())


def _op_sim_continue(r: Runner, p):
    # rebind: end_at -> max_iteration, result -> md_loop_continue
    r.set("result", int(r.get("timestep", 0)) <= int(r.get("end_at", 0)))


_OPS = {
    "global": _op_global,
    "species": _op_species,
    "particle_types": _op_particle_types,
    "particle_type_add_properties": _op_particle_type_add_properties,
    "domain": _op_domain,
    "lattice": _op_lattice,
    "bulk_lattice": _op_lattice,
    "gaussian_noise_r": _op_gaussian_noise_r,
    "gaussian_noise_v": _op_gaussian_noise_v,
    "init_rcut_max": _op_init_rcut_max,
    "init_particles": _op_init_particles,
    "chunk_neighbors": _op_chunk_neighbors,
    "nbh_dist": _op_nbh_dist,
    "particle_displ_over": _op_particle_displ_over,
    "particle_displ_over_async_end": _op_particle_displ_over_async_end,
    "lj_compute_force": _op_lj,
    "lj_compute_force_symetric": _op_lj_symetric,
    "lj_multi_force": _op_lj_multi,
    "lj_plot": _op_lj_plot,
    "eam_alloy_init": _op_eam_alloy_init,
    "eam_alloy_force": _op_eam_alloy_force,
    "johnson_force": _op_johnson,
    "johnson_emb": lambda r, p: _op_johnson(r, p, "johnson_emb"),
    "johnson_force_reuse_emb": lambda r, p: _op_johnson(r, p, "johnson_force_reuse_emb"),
    "johnson_init": _op_johnson_init,
    "zero_force_energy": _op_zero,
    "force_to_accel": _op_accel,
    "push_f_v_r": _op_push_f_v_r,
    "push_f_v": _op_push_f_v,
    "trigger_thermostate_screen": _op_trigger_screen,
    "trigger_thermostate_file": _op_trigger_file,
    "trigger_thermostate_compute": lambda r, p: None,
    "thermostate_compute_if_triggered": _op_thermo_compute_if,
    "thermostate_screen_if_triggered": _op_thermo_screen_if,
    "thermostate_file_if_triggered": _op_thermo_file_if,
    "default_thermostate_compute": _op_default_thermo_compute,
    "default_thermostate_screen": _op_default_thermo_screen,
    "default_thermostate_file": _op_default_thermo_file,
    "simulation_thermodynamic_state": _op_default_thermo_compute,
    "next_time_step": _op_next_time_step,
    "sim_continue": _op_sim_continue,
}


def parse_sets(argv):
    """--set-a-b value pairs -> ([a, b], value); other arguments pass through."""
    sets, rest = [], []
    it = iter(argv)
    for a in it:
        if a.startswith("--set-"):
            try:
                v = next(it)
            except StopIteration:
                raise DeckError(f"{a} needs a value") from None
            sets.append((a[len("--set-"):].split("-"), v))
        else:
            rest.append(a)
    return sets, rest


def main(argv=None):
    sets, rest = parse_sets(list(sys.argv[1:] if argv is None else argv))
    ap = argparse.ArgumentParser(description="Run an exaStamp deck (force-path subset) on one GPU.")
    ap.add_argument("deck")
    ap.add_argument("--config-dir", action="append", default=[], help="extra include / table search directory")
    ap.add_argument("--mixed", action="store_true", help="FP32 pair and spline math (XS_MIXED)")
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--thermo-file", default=None)
    a = ap.parse_args(rest)
    cfg = load_deck(a.deck, a.config_dir, sets)
    Runner(cfg, mixed=a.mixed, seed=a.seed, thermo_file=a.thermo_file).run()
    return 0


if __name__ == "__main__":
    sys.exit(main())
