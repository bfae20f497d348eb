"""Workloads of the marker-in-cell transfer framework: what a program built on it has it do, over
the range of grids and marker counts it is used for.

Kinds of a case (each through the package's public entry points):
  step       one resident transfer step (Context.step_transfer): marker properties, scatter, node
             properties, both assemblies, gathers and RK4, everything staying in HBM
  timestep   one whole resident timestep, the reaction, viscosity, porosity, melt composition,
             pressure back-trace and replenishment included, each by its own call
  plastic    one plastic iteration of the solver hand-off: new viscosities to the device, the
             Stokes-Darcy assembly, the pattern query and the fetch that the solver needs
  functions  the transfer functions one by one on host arrays (the drop-in boundary)
  adjoint    the checkpointed gradient of sum(tk1^2) with respect to the initial markers
  pullback   the reverse-mode functions on host arrays

A case: Nx x Ny basic nodes of a box of the given size, mcx x mcy markers a cell (jittered lattice,
planetesimal in sticky air), the property mode of src/constants.jl and the precision form.

A program that steps in HBM reads its state back when it wants it, not after every step, so the
outputs of the resident kinds are read from the device when they are looked at (Resident).  A
matrix is given as the dense table of its rows' stencil entries (_stencil_table): which entries
that cancel to zero are stored follows the last bit of the node sums.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "erebus.jl_amd"))

import ereb  # noqa: E402
from ereb import api, synth  # noqa: E402

START_TIME = 2.25e6 * 365.25 * 24 * 3600  # s, the reference's start time
DT = ereb.DT_LONGEST
DEV = "cuda" if torch.cuda.is_available() else "cpu"

PROPS = ["rhototalm", "rhocptotalm", "etatotalm", "hrtotalm", "ktotalm", "tkm_rhocptotalm",
         "etafluidcur_inv_kphim"]
STATE = ["xm", "ym", "tkm", "sxxm", "sxym"]
TYPED = {"inv_gggtotalm": "gggsolidm", "fricttotalm": "frictsolidm", "cohestotalm": "cohessolidm",
         "tenstotalm": "tenssolidm", "rhofluidcur": "rhofluidm", "alphasolidcur": "alphasolidm",
         "alphafluidcur": "alphafluidm"}
# SUM grids of each staggered grid: (values summed, names); the last one sums the weights
SUMMED = {
    "basic": ["etatotalm", "etavpm", "inv_gggtotalm", "sxym", "cohestotalm", "tenstotalm",
              "fricttotalm", None],
    "vx": ["rhototalm", "rhofluidcur", "ktotalm", "phim", "etafluidcur_inv_kphim", None],
    "vy": ["rhototalm", "rhofluidcur", "ktotalm", "phim", "etafluidcur_inv_kphim", None],
    "p": ["rhototalm", "rhocptotalm", "alphasolidcur", "alphafluidcur", "hrtotalm",
          "inv_gggtotalm", "sxxm", "tkm_rhocptotalm", "phim", None],
}
NODES = {
    "basic": ["ETA0", "ETA", "GGG", "SXY0", "COH", "TEN", "FRI"],
    "vx": ["RHOX", "RHOFX", "KX", "PHIX", "RX"],
    "vy": ["RHOY", "RHOFY", "KY", "PHIY", "RY"],
    "p": ["RHO", "RHOCP", "ALPHA", "ALPHAF", "HR", "GGGP", "SXX0", "tk1", "PHI", "BETAPHI"],
}
SUM_NAMES = {"basic": ereb.SUM_FIELDS[:8], "vx": ereb.SUM_FIELDS[8:14],
             "vy": ereb.SUM_FIELDS[14:20], "p": ereb.SUM_FIELDS[20:]}
INPUT_GRIDS = ["vx", "vy", "vxf", "vyf", "wyx", "ETAP", "ETAPHI", "gx", "gy", "DT", "tk2",
               "pr0", "pf0", "DMP", "HA", "HS", "DHP", "DSXX", "DSXY"]
SD_GRIDS = ["ETA", "ETAP", "GGG", "GGGP", "SXY0", "SXX0", "RHOX", "RHOY", "RHOFX", "RHOFY", "RX",
            "RY", "ETAPHI", "BETAPHI", "PHI", "gx", "gy", "pr0", "pf0", "DMP"]


def _case(name, kind, Nx, Ny, mcx, mcy, mode=1, form="fp64", box=140_000.0, **more):
    c = {"name": name, "kind": kind, "Nx": Nx, "Ny": Ny, "mcx": mcx, "mcy": mcy, "mode": mode,
         "form": form, "box": box, "planet": 0.357}
    c.update(more)
    return c


def listed():
    return [
        # the reference's test configuration: 3,136 markers, a step is its launches
        _case("step_15", "step", 15, 15, 4, 4, mode=9, box=14_000.0),
        # the reference's production configuration (141 x 141 nodes, 313,600 markers)
        _case("step_141", "step", 141, 141, 4, 4),
        # the benchmark workload, 2,822,400 markers, in both precision forms
        _case("step_281", "step", 281, 281, 6, 6),
        _case("step_281_mixed", "step", 281, 281, 6, 6, form="mixed"),
        # the largest workload of the benchmark, 20,070,400 markers
        _case("step_561", "step", 561, 561, 8, 8, planet=0.464),
        # a box with unequal sides, node counts that fill no tile and spacings that are not whole
        # metres, unequal marker counts along the two axes
        _case("step_173x97", "step", 173, 97, 5, 7, box=100_000.0),
        # every row of a timestep, at the million-marker workload
        _case("timestep_201", "timestep", 201, 201, 5, 5),
        # a plastic iteration of the benchmark grid, handed to a host solver
        _case("plastic_281", "plastic", 281, 281, 6, 6),
        # the functions one by one from host arrays, production configuration
        _case("functions_141", "functions", 141, 141, 4, 4),
        # the gradient of 5 steps of a small model and of the benchmark's 20 steps
        _case("adjoint_41", "adjoint", 41, 41, 5, 5, steps=5, every=5),
        _case("adjoint_201", "adjoint", 201, 201, 5, 5, steps=20, every=5),
        # the reverse-mode functions of a small model from host arrays
        _case("pullback_41", "pullback", 41, 41, 5, 5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "timestep", "plastic", "functions", "adjoint",
                       "pullback"])
    hi = {"step": 560, "timestep": 300, "plastic": 400, "functions": 200, "adjoint": 200,
          "pullback": 90}[kind]
    N = _log(rng, 15, hi)
    ratio = rng.uniform(0.6, 1.0)  # unequal sides
    Nx, Ny = (N, max(11, int(N * ratio))) if rng.random() < 0.5 else (max(11, int(N * ratio)), N)
    mcx, mcy = rng.randint(3, 7), rng.randint(3, 7)
    form = "mixed" if kind == "step" and rng.random() < 0.35 else "fp64"
    more = {"planet": round(rng.uniform(0.2, 0.45), 3)}
    if kind == "adjoint":
        more["steps"] = rng.randint(2, 15)
        more["every"] = rng.randint(2, 5)
        mcx, mcy = min(mcx, 5), min(mcy, 5)
    c = _case("", kind, Nx, Ny, mcx, mcy, mode=rng.choice([1, 1, 9]), form=form,
              box=float(rng.choice([14_000.0, 100_000.0, 140_000.0])), **more)
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------


def _geometry(case):
    Nx, Ny = case["Nx"], case["Ny"]
    side = max(Nx, Ny) - 1
    xs, ys = case["box"] * (Nx - 1) / side, case["box"] * (Ny - 1) / side
    R = case["planet"] * min(xs, ys)
    g = ereb.Geometry(Nx=Nx, Ny=Ny, xsize=xs, ysize=ys, Nxmc=case["mcx"], Nymc=case["mcy"],
                      rplanet=R, rcrust=0.96 * R)
    return g, ereb.Materials(marker_property_mode=case["mode"])


def _markers(g, mat, seed):
    """Marker vectors (torch, float64, on the GPU): a jittered lattice in column-major order, a
    porous partly hydrated planetesimal with random temperatures and stresses, sticky air."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    nx, ny = g.Nxm, g.Nym
    M = nx * ny

    def u():
        return torch.rand(M, generator=gen, device=DEV, dtype=torch.float64)

    m = torch.arange(M, device=DEV)
    jm, im = torch.div(m, ny, rounding_mode="floor").double(), (m % ny).double()
    x = g.dxm / 2 + jm * g.dxm + (u() - 0.5) * g.dxm
    y = g.dym / 2 + im * g.dym + (u() - 0.5) * g.dym
    r = torch.hypot(x - g.xcenter, y - g.ycenter)
    rock = r < g.rplanet
    tm = torch.where(rock, torch.where(r > g.rcrust, 2, 1), 3)

    def tab(name):
        return torch.tensor(getattr(mat, name), dtype=torch.float64, device=DEV)[tm - 1]

    def air(v):
        return torch.where(rock, 0.0, v)

    d = {"xm": x, "ym": y, "tm": tm,
         "phim": torch.where(rock, 0.05 + 0.25 * u(), mat.phimin),
         "tkm": torch.where(rock, 150.0 + 150.0 * u(), 273.0),
         "sxxm": torch.where(rock, 1e4 * (u() - 0.5), 0.0),
         "sxym": torch.where(rock, 1e4 * (u() - 0.5), 0.0),
         "XWsolidm0": torch.where(rock, 0.2 + 0.6 * u(), 0.0),
         "etavpm": tab("etasolidm")}
    for f, t in TYPED.items():
        d[f] = 1.0 / tab(t) if f == "inv_gggtotalm" else tab(t)
    d["rhototalm"] = air(tab("rhosolidm"))
    d["rhocptotalm"] = air(tab("rhocpsolidm"))
    d["etatotalm"] = air(tab("etasolidm"))
    d["hrtotalm"] = air(tab("start_hrsolidm"))
    d["ktotalm"] = air(tab("ksolidm"))
    return d


def _host(d):
    return {k: v.cpu().numpy() for k, v in d.items()}


def _grids(g, mat, seed):
    """The grids that the solves and the grid-only rows of a timestep produce."""
    rng = np.random.default_rng(int(seed) + 77)
    ph = rng.uniform(0.0, math.pi, 12)
    S, B = g.stag_shape, g.basic_shape
    vx, vy = synth.stream_velocity(g)
    vmax = max(np.abs(vx).max(), np.abs(vy).max())
    d = {"vx": vx, "vy": vy,
         "vxf": np.asfortranarray(vx + synth.smooth_field(g, S, 0.1 * vmax, 3, 2, ph[0])),
         "vyf": np.asfortranarray(vy + synth.smooth_field(g, S, 0.1 * vmax, 2, 3, ph[1])),
         "wyx": synth.rotation_rate(g, vx, vy)}
    d["gx"], d["gy"] = synth.disk_gravity(g)
    a = g.axes()
    X, Y = np.meshgrid(a["xp"], a["yp"])
    rock = np.hypot(X - g.xcenter, Y - g.ycenter) < g.rplanet
    d["ETAP"] = np.asfortranarray(np.where(rock, 1e19, 1e16))
    d["ETAPHI"] = np.asfortranarray(d["ETAP"] / np.where(rock, 0.175, 1e-4))
    d["tk2"] = np.asfortranarray(np.where(rock, 230.0, 273.0)
                                 + synth.smooth_field(g, S, 5.0, 2, 1, ph[2]))
    d["DT"] = synth.smooth_field(g, S, 1e-4, 2, 1, ph[3])
    d["pr0"] = mat.psurface + synth.smooth_field(g, S, 1e5, 1, 1, ph[4])
    d["pf0"] = mat.psurface + synth.smooth_field(g, S, 9e4, 1, 1, ph[5])
    for n in ("DMP", "HA", "HS", "DHP"):
        d[n] = np.zeros(S, order="F")
    d["DSXX"] = synth.smooth_field(g, S, 10.0, 3, 2, ph[6])
    d["DSXY"] = synth.smooth_field(g, B, 10.0, 2, 3, ph[7])
    return d


def _timestep_grids(g, mat, seed):
    rng = np.random.default_rng(int(seed) + 78)
    S, B = g.stag_shape, g.basic_shape
    d = {"YNY_inv_ETA": np.asfortranarray(1e-19 * (1 + rng.random(B))),
         "APHI": np.asfortranarray(1e-14 * (rng.random(S) - 0.5))}
    for n in ("pf", "pr", "ps"):
        d[n] = np.asfortranarray(mat.psurface + 1e5 * rng.random(S))
    return d, np.asfortranarray((rng.random(B) < 0.3).astype(np.uint8))


def _plastic_grids(g, mat, seed):
    """The 20 grids of the Stokes-Darcy assembly, constant in the air, and the viscosities of a
    second iteration."""
    rng = np.random.default_rng(int(seed) + 79)
    a = g.axes()
    S, B = g.stag_shape, g.basic_shape

    def inside(xs, ys):
        X, Y = np.meshgrid(xs, ys)
        return np.hypot(X - g.xcenter, Y - g.ycenter) < g.rplanet

    b, vx, vy, p = (inside(a["x"], a["y"]), inside(a["xvx"], a["yvx"]),
                    inside(a["xvy"], a["yvy"]), inside(a["xp"], a["yp"]))

    def mix(where, shape, rock, spread, air):
        return np.asfortranarray(np.where(where, rock * (1 + spread * rng.random(shape)), air))

    d = {"ETA": mix(b, B, 1e19, 0.5, 1e16), "ETAP": mix(p, S, 1e19, 0.5, 1e16),
         "GGG": mix(b, B, 1e10, 0.0, 1e10), "GGGP": mix(p, S, 1e10, 0.0, 1e10),
         "SXY0": mix(b, B, 1e4, 1.0, 0.0), "SXX0": mix(p, S, 1e4, 1.0, 0.0),
         "RHOX": mix(vx, S, 3000.0, 0.1, 1.0), "RHOY": mix(vy, S, 3000.0, 0.1, 1.0),
         "RHOFX": mix(vx, S, 1000.0, 0.0, 1.0), "RHOFY": mix(vy, S, 1000.0, 0.0, 1.0),
         "RX": mix(vx, S, 1e25, 1.0, 1e20), "RY": mix(vy, S, 1e25, 1.0, 1e20),
         "ETAPHI": mix(p, S, 5e19, 0.5, 1e20), "BETAPHI": mix(p, S, 1e-11, 0.5, 1e-14),
         "PHI": mix(p, S, 0.15, 0.5, 1e-4),
         "pr0": mat.psurface + synth.smooth_field(g, S, 1e5, 1, 1),
         "pf0": mat.psurface + synth.smooth_field(g, S, 9e4, 1, 1),
         "DMP": np.zeros(S, order="F")}
    d["gx"], d["gy"] = synth.disk_gravity(g)
    return d, mix(b, B, 1e18, 2.0, 1e16)


class Resident(dict):
    """Outputs that stay in the context's memory: an entry is read when it is looked at."""

    def __init__(self, readers):
        super().__init__((k, None) for k in readers)
        self._readers = readers

    def __getitem__(self, k):
        return self._readers[k]()


def _stencil_table(g, per_cell, colptr, rowval, nzval):
    """Rows of a CSC matrix as a dense (row, stencil entry) table: the unknowns of the 3 x 3 cells
    around the row's cell, absent entries 0."""
    n = colptr.size - 1
    col = np.repeat(np.arange(n, dtype=np.int64), np.diff(colptr))
    row = np.asarray(rowval) - 1
    rc, cc = row // per_cell, col // per_cell
    dj = cc // g.Ny1 - rc // g.Ny1 + 1
    di = cc % g.Ny1 - rc % g.Ny1 + 1
    out = np.zeros((n, 9 * per_cell))
    out[row, (dj * 3 + di) * per_cell + col % per_cell] = nzval
    return out


def _system_readers(g, ctx):
    def table(which, per_cell):
        cp, rv, nz, _ = ctx.csc(which)
        return _stencil_table(g, per_cell, cp, rv, nz)

    return {"L": lambda: table(ereb.SYS_STOKES_DARCY, 6), "LT": lambda: table(ereb.SYS_THERMAL, 1),
            "R": lambda: ctx.csc(ereb.SYS_STOKES_DARCY, pattern=False)[3],
            "RT": lambda: ctx.csc(ereb.SYS_THERMAL, pattern=False)[3]}


def _field_readers(ctx, markers, grids):
    r = {f: (lambda f=f: ctx.get_marker(f)) for f in markers}
    r.update({n: (lambda n=n: ctx.get_grid(n)) for n in grids})
    return r


def _node_readers(ctx):
    r = _field_readers(ctx, [], [n for k in NODES for n in NODES[k]])
    for k, names in SUM_NAMES.items():
        r["sums_" + k] = lambda names=names: np.stack([ctx.get_grid(n) for n in names])
    r["YNY"] = ctx.get_yny
    return r


def prepare(case, seed):
    kind = case["kind"]
    g, mat = _geometry(case)
    hrs, hrf = mat.radioactive_heating(START_TIME)
    s = {"kind": kind, "g": g, "mat": mat, "mode": case["mode"], "hrs": hrs, "hrf": hrf, "n": 0}
    ctx = s["ctx"] = ereb.Context(g, mat, ereb.MIXED if case["form"] == "mixed" else ereb.FP64)
    if kind == "plastic":
        grids, eta2 = _plastic_grids(g, mat, seed)
        for n in SD_GRIDS:
            ctx.set_grid(n, grids[n])
        s["eta"] = [eta2, grids["ETA"]]
        n, cap = 6 * g.Ny1 * g.Nx1, 44 * g.Ny1 * g.Nx1
        s["out"] = (ctx.host_array(n + 1, np.int64), ctx.host_array(cap, np.int64),
                    ctx.host_array(cap, np.float64), ctx.host_array(n, np.float64))
        return s
    mk = _host(_markers(g, mat, seed))
    if kind in ("step", "timestep"):
        ctx.set_markers(mk)
        grids = _grids(g, mat, seed)
        for n in INPUT_GRIDS:
            ctx.set_grid(n, grids[n])
        s["read"] = _field_readers(ctx, STATE + PROPS, [])
        s["read"].update(_node_readers(ctx))
        s["read"].update(_system_readers(g, ctx))
        if kind == "timestep":
            more, yny = _timestep_grids(g, mat, seed)
            for n, a in more.items():
                ctx.set_grid(n, a)
            ctx.set_yny(yny)
            s["hyd"] = ereb.Hydration()
            ctx.set_marker("XWsolidm", mk["XWsolidm0"])
            ctx.set_marker("phinewm", mk["phim"])
            ctx.set_marker("pfm0", np.zeros(mk["xm"].size))
            # WTPSUM and YNY are written by several rows: their last values
            s["read"].update(_field_readers(
                ctx, ["phim", "etavpm", "XWsolidm", "phinewm", "pfm0"],
                ["XWS", "DMP", "DHP", "pr0", "pf0", "ps0"]))
        ctx.sync()
    elif kind == "adjoint":
        ctx.set_markers(mk)
        vx, vy = synth.stream_velocity(g)
        for n, a in (("vx", vx), ("vy", vy), ("vxf", vx), ("vyf", vy),
                     ("wyx", np.zeros(g.basic_shape, order="F"))):
            ctx.set_grid(n, a)
        M = mk["xm"].size
        s["steps"], s["every"] = case["steps"], case["every"]
        s["out"] = (ctx.host_array(M, np.float64), ctx.host_array(M, np.float64))
    elif kind == "functions":
        s["mk"], s["gr"] = mk, _grids(g, mat, seed)
        M = mk["xm"].size
        for f in PROPS[5:]:
            mk[f] = np.zeros(M)
        s["sums"] = [np.zeros(g.basic_shape if k < 8 else g.stag_shape, order="F")
                     for k in range(30)]
        s["node"] = {n: np.zeros(g.basic_shape if k == "basic" else g.stag_shape, order="F")
                     for k in NODES for n in NODES[k]}
        s["node"]["YNY"] = np.zeros(g.basic_shape, dtype=np.uint8, order="F")
        s["R"], s["RT"] = np.zeros(6 * g.Ny1 * g.Nx1), np.zeros(g.Ny1 * g.Nx1)
    else:  # pullback
        s["mk"], s["gr"] = mk, _grids(g, mat, seed)
        s["bar"] = _cotangents(g, mk["xm"].size, seed)
    return s


def _cotangents(g, M, seed):
    rng = np.random.default_rng(int(seed) + 80)

    def grid(shape):
        return np.asfortranarray(rng.uniform(-1.0, 1.0, shape))

    return {"sums": [grid(g.basic_shape if k < 8 else g.stag_shape) for k in range(30)],
            "props": [rng.uniform(-0.5, 0.5, M) for _ in range(7)],
            "rk4": {k: rng.uniform(-0.5, 0.5, M) * (1e-3 if k in ("xm", "ym") else 1.0)
                    for k in ("xm", "ym", "tkm", "sxym", "sxxm")}}


# ---- one pass ------------------------------------------------------------------


def _dt(s):
    """dt of this pass.  Every second pass goes back in time, so that the markers of a state that is
    stepped any number of times stay those of a timestep (each pass moves them by the same half
    cell)."""
    s["n"] += 1
    return DT if s["n"] % 2 else -DT


def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "step":
        ctx.step_transfer(s["hrs"], s["hrf"], s["mode"], _dt(s), 2)
        return Resident(s["read"])
    if kind == "timestep":
        dt, hyd = _dt(s), s["hyd"]
        ctx.step_scatter(s["hrs"], s["hrf"], s["mode"])
        ctx.step_node_properties()
        ctx.step_thermochemical_reaction(DT, 2, 3, hyd=hyd)
        ctx.step_assemble_stokes_darcy(dt)
        ctx.step_assemble_thermal(dt)
        ctx.step_marker_viscosity()
        ctx.step_gather_stress()
        ctx.step_gather_temperature(2)
        ctx.step_marker_porosity(dt, hyd=hyd)
        ctx.step_melt_composition()
        ctx.step_advect_rk4(dt, s["mode"])
        ctx.step_backtrace_pressures(dt)
        ctx.step_replenish_markers(maps=False)
        return Resident(s["read"])
    if kind == "plastic":
        s["n"] += 1
        which = ereb.SYS_STOKES_DARCY
        ctx.set_grid("ETA", s["eta"][s["n"] % 2])
        ctx.step_assemble_stokes_darcy(DT)
        fetch = s["out"] if ctx.csc_pattern_changed(which) else (None, None) + s["out"][2:]
        got = ctx.csc(which, out=fetch)
        n, nnz = got[3].size, got[2].size
        return _page_locked(s, {"colptr": s["out"][0][:n + 1], "rowval": s["out"][1][:nnz],
                                "nzval": got[2], "R": got[3]})
    if kind == "adjoint":
        L, gT, gP, _ = ctx.adjoint_tk1_loss(s["steps"], s["every"], DT, s["mode"], s["hrs"],
                                            s["hrf"], out=s["out"])
        return _page_locked(s, {"loss": L, "tkm": gT, "phim": gP})
    if kind == "functions":
        return _run_functions(s)
    return _run_pullback(s)


def _page_locked(s, arrays):
    """Outputs in the page-locked arrays of a context, which live as long as it: `s` is kept."""
    return Resident({k: (lambda a=a, s=s: a if isinstance(a, float) else np.array(a))
                     for k, a in arrays.items()})


def _run_functions(s):
    ctx, g, mk, gr, nd = s["ctx"], s["g"], s["mk"], s["gr"], s["node"]
    M, dt, sums = mk["xm"].size, _dt(s), s["sums"]
    api.marker_to_nodes_(
        ctx, *[mk[f] for f in ("xm", "ym", "tm", "tkm", "phim", "XWsolidm0", "etavpm",
                               "inv_gggtotalm", "fricttotalm", "cohestotalm", "tenstotalm",
                               "rhofluidcur", "alphasolidcur", "alphafluidcur", "sxxm", "sxym")],
        *[mk[f] for f in PROPS], s["hrs"], s["hrf"], s["mode"], sums, M)
    api.compute_basic_node_properties_(ctx, *sums[:8], *[nd[n] for n in NODES["basic"]], nd["YNY"])
    api.compute_vx_node_properties_(ctx, *sums[8:14], *[nd[n] for n in NODES["vx"]])
    api.compute_vy_node_properties_(ctx, *sums[14:20], *[nd[n] for n in NODES["vy"]])
    api.compute_p_node_properties_(ctx, *sums[20:], *[nd[n] for n in NODES["p"]])
    api.apply_insulating_boundary_conditions_(ctx, nd["tk1"])
    both = {**gr, **nd}
    L = api.assemble_hydromechanical_lse_(ctx, *[both[n] for n in SD_GRIDS], dt, s["R"])
    LT = api.assemble_thermal_lse_(ctx, nd["tk1"], nd["RHOCP"], nd["KX"], nd["KY"], nd["HR"],
                                   gr["HA"], gr["HS"], gr["DHP"], s["RT"], dt)
    api.update_marker_stress_(ctx, mk["xm"], mk["ym"], mk["sxxm"], mk["sxym"], gr["DSXX"],
                              gr["DSXY"], M)
    api.update_marker_temperature_(ctx, mk["xm"], mk["ym"], mk["tkm"], gr["DT"], gr["tk2"], 2, M)
    api.move_markers_rk4_(ctx, mk["xm"], mk["ym"], mk["tm"], mk["tkm"], mk["phim"], mk["sxym"],
                          mk["sxxm"], gr["vx"], gr["vy"], gr["vxf"], gr["vyf"], gr["wyx"],
                          gr["tk2"], M, dt, s["mode"])
    read = {f: (lambda f=f: mk[f]) for f in STATE + PROPS}
    read.update({n: (lambda n=n: nd[n]) for n in nd})
    at = 0
    for k, names in SUM_NAMES.items():
        read["sums_" + k] = lambda a=at, b=at + len(names): np.stack(sums[a:b])
        at += len(names)
    read["L"] = lambda: _stencil_table(g, 6, L.colptr, L.rowval, L.nzval)
    read["LT"] = lambda: _stencil_table(g, 1, LT.colptr, LT.rowval, LT.nzval)
    read["R"], read["RT"] = (lambda: s["R"]), (lambda: s["RT"])
    return Resident(read)


def _run_pullback(s):
    ctx, mk, gr, bar = s["ctx"], s["mk"], s["gr"], s["bar"]
    M = mk["xm"].size
    out = {"nodes": api.marker_to_nodes_pullback(ctx, mk, s["hrs"], s["hrf"], s["mode"],
                                                 bar["sums"], bar["props"])}
    t = api.update_marker_temperature_pullback(ctx, mk["xm"], mk["ym"], gr["DT"], gr["tk2"], 2, M,
                                               bar["rk4"]["tkm"])
    out["temperature"] = dict(zip(("tkm", "DT", "tk2", "xm", "ym"), t))
    t = api.update_marker_stress_pullback(ctx, mk["xm"], mk["ym"], gr["DSXX"], gr["DSXY"], M,
                                          bar["rk4"]["sxxm"], bar["rk4"]["sxym"])
    out["stress"] = dict(zip(("DSXX", "DSXY", "xm", "ym"), t))
    mo, go = api.move_markers_rk4_pullback(
        ctx, mk["xm"], mk["ym"], mk["tm"], mk["tkm"], mk["phim"], mk["sxym"], mk["sxxm"], gr["vx"],
        gr["vy"], gr["vxf"], gr["vyf"], gr["wyx"], gr["tk2"], M, DT, s["mode"], bar["rk4"])
    out["rk4"], out["rk4_grids"] = mo, go
    return out


def work(case):
    """Bytes: each marker vector and grid that the functions take read once, each they give written
    once (Float64 8, the mixed form's property vectors 4, marker types 4, matrix entries 12);
    operations of the arithmetic per marker and cell."""
    g, _ = _geometry(case)
    M, N = g.Nxm * g.Nym, g.Nx1 * g.Ny1
    p = 4 if case["form"] == "mixed" else 8
    # r xm ym tkm phim sxx sxy (8) tm (4) XW etavp 7 material (p); w xm ym tkm sxx sxy, 7 properties
    step_m = 6 * 8 + 4 + 9 * p + 5 * 8 + 7 * p
    # r 19 grids, w 30 SUM + 27 node grids, R, RT; ~38 + 5 entries a cell in both matrices
    step_n = (19 + 57 + 6 + 1) * 8 + 43 * 12
    kind = case["kind"]
    if kind in ("step", "functions"):
        return {"bytes": M * step_m + N * step_n, "flops": M * 1300.0 + N * 600.0}
    if kind == "timestep":
        # + viscosity (tm tkm -> etatotal etavp), reaction, porosity, XW, and their grids
        return {"bytes": M * (step_m + 2 * 8 + 6 * 8 + 8 + 8) + N * (step_n + 20 * 8),
                "flops": M * 1600.0 + N * 800.0}
    if kind == "plastic":
        return {"bytes": N * (20 * 8 + 6 * 8 + 38 * 8.0), "flops": N * 500.0}
    if kind == "adjoint":
        # a step of the differentiated map: scatter and RK4, and about twice that backwards
        m, n = 6 * 8 + 4 + 9 * 8 + 5 * 8, (10 + 27) * 8
        return {"bytes": case["steps"] * 3.0 * (M * m + N * n), "flops": case["steps"] * M * 4000.0}
    return {"bytes": M * (23 + 7 + 20 + 4 + 5 + 5 + 12 + 16) * 8.0 + N * 60 * 8.0,
            "flops": M * 4000.0}


# ---- the same in plain torch, 64 bits ---------------------------------------------


class _Plain:
    """The transfer functions on one geometry as plain torch operations; differentiable."""

    def __init__(self, g, mat, mode):
        self.g, self.mat, self.mode = g, mat, mode
        self.idx, self.idy = 1.0 / g.dx, 1.0 / g.dy
        half = {"basic": (0, 0), "vx": (0, 1), "vy": (1, 0), "p": (1, 1)}
        # first node, clamps of the cell column and row
        self.spec = {k: (-g.dx / 2 * hx, -g.dy / 2 * hy, g.Nx - 1 + hx, g.Ny - 1 + hy)
                     for k, (hx, hy) in half.items()}

    def cell(self, k, x, y, lo=1, hi=0):
        """0-based column and row of the cell and the distances from its first node, in cells."""
        x0, y0, jm, im = self.spec[k]
        g = self.g
        j = ((x.detach() - x0) * self.idx).trunc().clamp(lo - 1, jm - 1 - hi)
        i = ((y.detach() - y0) * self.idy).trunc().clamp(lo - 1, im - 1 - hi)
        return j.long(), i.long(), (x - (x0 + j * g.dx)) / g.dx, (y - (y0 + i * g.dy)) / g.dy

    @staticmethod
    def weights(a, b):
        return (1 - b) * (1 - a), b * (1 - a), (1 - b) * a, b * a

    def rows(self, k):
        return self.g.Ny if k == "basic" else self.g.Ny1

    def at(self, k, grid, i, j):
        return grid[j * self.rows(k) + i]  # grids flat, column-major

    def interp(self, k, grid, x, y, lo=1, hi=0):
        j, i, a, b = self.cell(k, x, y, lo, hi)
        w = self.weights(a, b)
        at = [self.at(k, grid, i + di, j + dj) for dj in (0, 1) for di in (0, 1)]
        return sum(v * q for v, q in zip(at, w))

    def tab(self, name, tm):
        v = getattr(self.mat, name) if isinstance(name, str) else name
        return torch.tensor(np.asarray(v), dtype=torch.float64, device=tm.device)[tm - 1]

    def rhocpf(self, T):
        m = self.mat
        if self.mode == 9:
            return torch.full_like(T, m.rhocpfluidm[0])
        tf, ri, rw = m.tmfluidphase, m.rhoH2Ofi, m.rhoH2Of
        hot = rw * (-4.67e4 + 333.0 * T - 0.731 * T * T + 5.4e-4 * T * T * T)
        r = torch.where(T < 410.0, rw * 4200.0, hot)
        r = torch.where(T < tf + 5.0, rw * (4200.0 + 0.1 * m.Lf), r)
        r = torch.where(T < tf, ri * (7.67 * T + 0.1 * m.Lf), r)
        return torch.where(T < tf - 5.0, ri * 7.67 * T, r)

    def properties(self, d, hrs, hrf):
        m, T, phi, XW, tm = self.mat, d["tkm"], d["phim"], d["XWsolidm0"], d["tm"]
        rock = tm < 3

        def total(s, f):
            return s * (1 - phi) + f * phi

        if self.mode == 9:
            ks, kf = torch.full_like(T, m.ksolidm[0]), torch.full_like(T, m.kfluidm[0])
        else:
            ks = 0.73 + 1293.0 / (T + 77.0)
            kf = torch.where(T < 410.0, -0.581 + 6.34e-3 * T - 7.93e-6 * T * T,
                             -0.142 + 4.12e-3 * T - 5.01e-6 * T * T)
            kf = torch.where(T < m.tmfluidphase, 0.465 + 488.0 / T, kf)
        t = ks * (3 * phi - 2) + kf * (1 - 3 * phi)
        k = torch.sqrt(ks * kf / 2 + t * t / 16) - t / 4
        rhos = (m.MD + m.MH2O * XW) / (m.VDs * (1 - XW) + m.VWs * XW)
        warm = T > m.tmfluidphase
        rhof = torch.where(warm, m.rhoH2Of, m.rhoH2Ofi)
        es = torch.where(T > m.tmsolidphase, self.tab("etasolidmm", tm), self.tab("etasolidm", tm))
        ef = torch.where(warm, self.tab("etafluidmm", tm), self.tab("etafluidm", tm))
        ef = torch.where(rock, ef, m.etafluidm[2])
        eta = torch.maximum(es.clamp(min=m.etamin), ef)
        p = {"rhototalm": total(rhos, rhof),
             "rhocptotalm": total(self.tab("rhocpsolidm", tm), self.rhocpf(T)),
             "etatotalm": eta, "hrtotalm": total(self.tab(hrs, tm), self.tab(hrf, tm)),
             "ktotalm": k}
        p = {f: torch.where(rock, v, d[f]) for f, v in p.items()}
        p["tkm_rhocptotalm"] = T * p["rhocptotalm"]
        q, r = m.phim0 / phi, (1 - phi) / (1 - m.phim0)
        p["etafluidcur_inv_kphim"] = ef / self.tab("kphim0", tm) * q ** 3 * r ** 2
        return p

    def sums(self, k, d, fields):
        """(number of fields, nodes) sums of value * weight; None sums the weights."""
        j, i, a, b = self.cell(k, d["xm"], d["ym"])
        rows, cols = self.rows(k), (self.g.Nx if k == "basic" else self.g.Nx1)
        w = self.weights(a, b)
        out = []
        for f in fields:
            acc = torch.zeros(rows * cols, dtype=torch.float64, device=a.device)
            for c in range(4):
                at = (j + c // 2) * rows + i + c % 2
                acc = acc.index_add(0, at, w[c] if f is None else w[c] * d[f])
            out.append(acc)
        return out

    def nodes(self, k, s):
        """Node grids from the SUM grids, 0 where no marker contributes."""
        ok = s[-1] > 0
        wt = torch.where(ok, s[-1], 1.0)

        def harm(v):
            return wt / torch.where(ok, v, 1.0)

        n = [v / wt for v in s[:-1]]
        if k == "basic":
            n[2] = harm(s[2])
        if k == "p":
            n[5] = harm(s[5])
            n[7] = s[7] / torch.where(ok, s[1], 1.0)
            n.append(n[8] / torch.where(ok, n[5], 1.0))
        return [torch.where(ok, v, 0.0) for v in n]

    def insulated(self, t):
        t = t.reshape(self.g.Nx1, self.g.Ny1)
        t = torch.cat([t[:, 1:2], t[:, 1:-1], t[:, -2:-1]], 1)
        return torch.cat([t[1:2], t[1:-1], t[-2:-1]], 0).reshape(-1)

    def stage(self, k, v, vc, x, y):
        """Velocity component at a marker: linear with the second-order correction along its own
        direction; `vc` gives the centre value of the first row's left-half correction."""
        j, i, a, b = self.cell(k, x, y)
        g = self.g

        def along(first, n, f, q):
            # node q of the row (or column) `first` and the corrected interpolation
            lo, hi = q(0), q(1)
            u = lo * (1 - f) + hi * f
            t = 0.5 * (f - 0.5) ** 2
            p = j if k == "vx" else i
            right = (f >= 0.5) & (p < n - 2)
            left = (f < 0.5) & (p > 0)
            mid = q(0, vc) if first else lo
            u = u + torch.where(right, t * (lo - 2 * hi + q(2)), 0.0)
            return u + torch.where(left, t * (q(-1) - 2 * mid + hi), 0.0)

        if k == "vx":
            def row(r, first):
                return along(first, g.Nx, a, lambda o, grid=v: self.at(
                    k, grid, i + r, (j + o).clamp(0, g.Nx)))
            return row(0, True) * (1 - b) + row(1, False) * b

        def colm(c, first):
            return along(first, g.Ny, b, lambda o, grid=v: self.at(
                k, grid, (i + o).clamp(0, g.Ny), j + c))
        return colm(0, True) * (1 - a) + colm(1, False) * a

    def rk4(self, d, gr, dt):
        c, b = (0.5, 0.5, 1.0), (1 / 6, 1 / 3, 1 / 3, 1 / 6)
        x0, y0 = d["xm"], d["ym"]
        tks0 = self.interp("p", gr["tk2"], x0, y0)
        th = dt * self.interp("basic", gr["wyx"], x0, y0)
        s, t = d["sxxm"], d["sxym"]
        out = {"sxxm": s * torch.cos(th) ** 2 - s * torch.sin(th) ** 2 - t * torch.sin(2 * th),
               "sxym": s * torch.sin(2 * th) + t * torch.cos(2 * th)}

        def trace(vx, vy, x, y, step):
            xr, yr, sx, sy = x, y, 0.0, 0.0
            for r in range(4):
                u, v = self.stage("vx", vx, gr["vx"], xr, yr), self.stage("vy", vy, vy, xr, yr)
                sx, sy = sx + b[r] * u, sy + b[r] * v
                if r < 3:
                    xr, yr = x + step * c[r] * u, y + step * c[r] * v
            return x + step * sx, y + step * sy

        x1, y1 = trace(gr["vx"], gr["vy"], x0, y0, dt)
        xf, yf = trace(gr["vxf"], gr["vyf"], x1, y1, -dt)
        dT = self.interp("p", gr["tk2"], xf, yf) - tks0
        T, ph = d["tkm"], d["phim"]
        rs, rf = self.tab("rhocpsolidm", d["tm"]), self.rhocpf(T)
        out.update(xm=x1, ym=y1, tkm=((1 - ph) * T * rs + ph * (T + dT) * rf)
                   / ((1 - ph) * rs + ph * rf))
        return out


def _exact_systems(g, mat, gr, nd, dt):
    """Both linear systems from the input grids and the node grids: stencil tables and right-hand
    sides."""
    rows, cols, dx, dy, K = g.Ny1, g.Nx1, g.dx, g.dy, mat.Kcont
    i, j = np.meshgrid(np.arange(1, rows + 1), np.arange(1, cols + 1), indexing="ij")

    def full(n):
        a = nd[n] if n in nd else gr[n]
        out = np.ones((rows + 2, cols + 2))  # a border, read by cells that don't use it
        out[1:1 + a.shape[0], 1:1 + a.shape[1]] = a
        return lambda di=0, dj=0: out[1 + di:1 + di + rows, 1 + dj:1 + dj + cols]

    A = {n: full(n) for n in SD_GRIDS + ["tk1", "RHOCP", "KX", "KY", "HR", "HA", "HS", "DHP"]}
    T, R = np.zeros((cols, rows, 6, 54)), np.zeros((cols, rows, 6))

    def put(eq, where, v, unknown, di=0, dj=0):
        at = T[:, :, eq, ((dj + 1) * 3 + di + 1) * 6 + unknown]
        at[where.T] = np.broadcast_to(v, i.shape).T[where.T]

    def rhs(eq, where, v):
        R[:, :, eq][where.T] = np.broadcast_to(v, i.shape).T[where.T]

    def maxwell(eta, ggg, s, di=0, dj=0):
        e, q = A[eta](di, dj), A[ggg](di, dj)
        return e * q * dt / (q * dt + e), A[s](di, dj) * e / (q * dt + e)

    with np.errstate(all="ignore"):
        for eq, (rho, gn, last, walls, sgn) in enumerate((
                ("RHOX", "gx", (j == g.Nx) | (j == cols), (mat.bc[2], mat.bc[3]), 1.0),
                ("RHOY", "gy", (i == g.Ny) | (i == rows), (mat.bc[0], mat.bc[1]), -1.0))):
            x = eq == 0
            edge = (i == 1) | (j == 1) | last | (i == rows if x else j == cols)
            h = (dx, dy) if x else (dy, dx)  # spacing along the component, and across

            def sh(along, across, x=x):
                return (across, along) if x else (along, across)  # (di, dj)

            e1, s1 = maxwell("ETA", "GGG", "SXY0", *sh(0, -1))
            e2, s2 = maxwell("ETA", "GGG", "SXY0")
            p1, n1 = maxwell("ETAP", "GGGP", "SXX0")
            p2, n2 = maxwell("ETAP", "GGGP", "SXX0", *sh(1, 0))
            r, gv = A[rho], A[gn]()
            da = 0.5 * (r(*sh(1, 0)) - r(*sh(-1, 0))) / h[0] * gv * dt
            db = 0.5 * (r(*sh(0, 1)) - r(*sh(0, -1))) / h[1] * gv * dt * 0.25
            ii = 1.0 / (dx * dy)
            one = ~edge
            put(eq, edge, 1.0, eq)
            inner = (1 < j) & (j < g.Nx) if x else (1 < i) & (i < g.Ny)
            put(eq, (i == 1 if x else j == 1) & inner, walls[0], eq, *sh(0, 1))
            put(eq, (i == rows if x else j == cols) & inner, walls[1], eq, *sh(0, -1))
            put(eq, one, p1 / h[0] ** 2, eq, *sh(-1, 0))
            put(eq, one, p2 / h[0] ** 2, eq, *sh(1, 0))
            put(eq, one, e1 / h[1] ** 2, eq, *sh(0, -1))
            put(eq, one, e2 / h[1] ** 2, eq, *sh(0, 1))
            put(eq, one, -(p1 + p2) / h[0] ** 2 - (e1 + e2) / h[1] ** 2 - da, eq)
            o = 1 - eq
            put(eq, one, (p1 - e2) * ii - db, o)
            put(eq, one, (e2 - p2) * ii - db, o, *sh(1, 0))
            put(eq, one, (e1 - p1) * ii - db, o, *sh(0, -1))
            put(eq, one, (p2 - e1) * ii - db, o, *sh(1, -1))
            put(eq, one, K / h[0], 2)
            put(eq, one, -K / h[0], 2, *sh(1, 0))
            rhs(eq, one, -r() * gv - (s2 - s1) / h[1] - sgn * (n2 - n1) / h[0])
            # Darcy flux along the same axis
            put(3 + eq, edge, 1.0, 3 + eq)
            fw = (mat.bcf[2], mat.bcf[3]) if x else (mat.bcf[0], mat.bcf[1])
            put(3 + eq, (i == 1 if x else j == 1) & inner, fw[0], 3 + eq, *sh(0, 1))
            put(3 + eq, (i == rows if x else j == cols) & inner, fw[1], 3 + eq, *sh(0, -1))
            put(3 + eq, one, A["RX" if x else "RY"](), 3 + eq)
            put(3 + eq, one, -K / h[0], 5)
            put(3 + eq, one, K / h[0], 5, *sh(1, 0))
            rhs(3 + eq, one, A["RHOFX" if x else "RHOFY"]() * gv)
        edge = (i == 1) | (i == rows) | (j == 1) | (j == cols)
        anchor = ~edge & ((i == 2) | (i == g.Ny) | (j == 2) | (j == g.Nx))
        one = ~edge & ~anchor
        phi, bp = A["PHI"](), A["BETAPHI"]()
        c = K / (1 - phi) * (1 / A["ETAPHI"]() + bp / dt)
        dp = (A["pr0"]() - A["pf0"]()) / (1 - phi) * bp / dt
        for eq, v, s, src in ((2, 0, 1.0, A["DMP"]()), (5, 3, -1.0, 0.0)):
            put(eq, edge, 1.0, eq)
            put(eq, anchor, K, eq)
            rhs(eq, anchor, mat.psurface)
            put(eq, one, -1 / dx, v, 0, -1)
            put(eq, one, 1 / dx, v)
            put(eq, one, -1 / dy, v + 1, -1, 0)
            put(eq, one, 1 / dy, v + 1)
            put(eq, one, s * c, 2)
            put(eq, one, -s * c, 5)
            rhs(eq, one, s * dp + src)
    L, Rv = T.reshape(-1, 54), R.reshape(-1)
    T, R = np.zeros((cols, rows, 1, 9)), np.zeros((cols, rows))
    for where, v, di, dj in (
            (edge, 1.0, 0, 0), (j == 1, -1.0, 0, 1), (j == cols, -1.0, 0, -1),
            ((i == 1) & (j > 1) & (j < cols), -1.0, 1, 0),
            ((i == rows) & (j > 1) & (j < cols), -1.0, -1, 0),
            (~edge, -A["KX"](0, -1) / dx ** 2, 0, -1), (~edge, -A["KX"]() / dx ** 2, 0, 1),
            (~edge, -A["KY"](-1, 0) / dy ** 2, -1, 0), (~edge, -A["KY"]() / dy ** 2, 1, 0),
            (~edge, A["RHOCP"]() / dt + (A["KX"](0, -1) + A["KX"]()) / dx ** 2
             + (A["KY"](-1, 0) + A["KY"]()) / dy ** 2, 0, 0)):
        at = T[:, :, 0, (dj + 1) * 3 + di + 1]
        at[where.T] = np.broadcast_to(v, i.shape).T[where.T]
    heat = A["RHOCP"]() / dt * A["tk1"]() + sum(A[n]() for n in ("HR", "HA", "HS", "DHP"))
    R[(~edge).T] = heat.T[(~edge).T]
    return {"L": L, "R": Rv, "LT": T.reshape(-1, 9), "RT": R.reshape(-1)}


def _flat(a):
    return torch.from_numpy(np.ascontiguousarray(a.ravel(order="F"))).to(DEV)


def _back(g, k, v):
    cols, rows = (g.Nx, g.Ny) if k == "basic" else (g.Nx1, g.Ny1)
    return np.asfortranarray(v.detach().cpu().numpy().reshape(cols, rows).T)


def exact(case, seed):
    kind = case["kind"]
    if kind == "plastic":
        return None
    g, mat = _geometry(case)
    hrs, hrf = mat.radioactive_heating(START_TIME)
    d = _markers(g, mat, seed)
    P = _Plain(g, mat, case["mode"])
    if kind == "adjoint":
        return _exact_adjoint(case, P, d, hrs, hrf)
    grids = _grids(g, mat, seed)
    gr = {n: _flat(a) for n, a in grids.items()}
    if kind == "pullback":
        return _exact_pullback(g, P, d, gr, hrs, hrf, _cotangents(g, d["xm"].numel(), seed))
    out = {"YNY": None}
    props = P.properties(d, hrs, hrf)
    full = {**d, **props}
    for k in SUMMED:
        s = P.sums(k, full, SUMMED[k])
        out["sums_" + k] = np.stack([_back(g, k, v) for v in s])
        for n, v in zip(NODES[k], P.nodes(k, s)):
            out[n] = _back(g, k, P.insulated(v) if n == "tk1" else v)
    out.update(_exact_systems(g, mat, grids, out, DT))
    if kind == "timestep":
        # the reaction's sums are in both right-hand sides, the later rows write WTPSUM again, the viscosity row etatotalm and etavpm
        out.update({f: None for f in ("R", "RT", "sums_p", "etatotalm", "etavpm", "XWsolidm", "phinewm",
                                      "pfm0", "XWS", "DMP", "DHP", "pr0", "pf0", "ps0")})
        props.pop("etatotalm")
        more, _ = _timestep_grids(g, mat, seed)
        a = P.interp("p", _flat(more["APHI"]), d["xm"], d["ym"])
        ph = d["phim"]
        new = (ph / ((1 - ph) * torch.exp(a * DT) + ph)).clamp(mat.phimin, 1 - mat.phimin)
        d["phim"] = torch.where(d["tm"] < 3, new, ph)
        out["phim"] = d["phim"].cpu().numpy()
    out.update({f: v.cpu().numpy() for f, v in props.items()})
    d["sxxm"] = d["sxxm"] + P.interp("p", gr["DSXX"], d["xm"], d["ym"], lo=2, hi=1)
    d["sxym"] = d["sxym"] + P.interp("basic", gr["DSXY"], d["xm"], d["ym"])
    d["tkm"] = d["tkm"] + P.interp("p", gr["DT"], d["xm"], d["ym"])
    out.update({f: v.cpu().numpy() for f, v in P.rk4(d, gr, DT).items()})
    return out


def _exact_adjoint(case, P, d, hrs, hrf):
    if case["steps"] * d["xm"].numel() > 25_000_000:  # the tape of a longer one is over the card
        return None
    vx, vy = synth.stream_velocity(P.g)
    gr = {"vx": _flat(vx), "vy": _flat(vy)}
    gr.update(vxf=gr["vx"], vyf=gr["vy"], wyx=_flat(np.zeros(P.g.basic_shape)))
    T0, ph = d["tkm"].clone().requires_grad_(), d["phim"].clone().requires_grad_()
    d = {**d, "tkm": T0, "phim": ph}
    for n in range(case["steps"] + 1):
        props = P.properties(d, hrs, hrf)
        s = P.sums("p", {**d, **props}, ["rhocptotalm", "tkm_rhocptotalm"])
        tk1 = P.insulated(torch.where(s[0] > 0, s[1] / torch.where(s[0] > 0, s[0], 1.0), 0.0))
        if n == case["steps"]:
            break
        d = {**d, **{f: props[f] for f in PROPS[:5]}}
        if n == 0:
            d["tkm"] = P.interp("p", tk1, d["xm"], d["ym"])
        moved = P.rk4(d, {**gr, "tk2": tk1}, DT)
        d.update(xm=moved["xm"], ym=moved["ym"], tkm=moved["tkm"])
    L = (tk1 * tk1).sum()
    gT, gP = torch.autograd.grad(L, (T0, ph), allow_unused=True)
    gT = torch.zeros_like(T0) if gT is None else gT
    return {"loss": float(L.detach()), "tkm": gT.cpu().numpy(), "phim": gP.cpu().numpy()}


def _exact_pullback(g, P, d, gr, hrs, hrf, bar):
    def leafs(names, src):
        return {n: src[n].clone().requires_grad_() for n in names}

    def grads(L, ins):
        got = torch.autograd.grad(L, list(ins.values()), allow_unused=True)
        return {n: torch.zeros_like(v) if q is None else q
                for (n, v), q in zip(ins.items(), got)}

    def as_grid(q, names, k=None):
        return {n: (_back(g, "basic" if n in ("wyx", "DSXY") else "p", v) if n in names
                    else v.cpu().numpy()) for n, v in q.items()}

    dev = {k: torch.from_numpy(v).to(DEV) for k, v in bar["rk4"].items()}
    ins = leafs([f for f in d if f != "tm"], d)
    full = {**d, **ins}
    props = P.properties(full, hrs, hrf)
    L = sum((torch.from_numpy(b).to(DEV) * props[f]).sum() for f, b in zip(PROPS, bar["props"]))
    at = 0
    for k in SUMMED:
        for v in P.sums(k, {**full, **props}, SUMMED[k]):
            L = L + (v * _flat(bar["sums"][at])).sum()
            at += 1
    out = {"nodes": {n: v.cpu().numpy() for n, v in grads(L, ins).items()}}
    ins = {**leafs(["xm", "ym"], d), **leafs(["DT", "tk2"], gr)}
    L = (dev["tkm"] * P.interp("p", ins["DT"], ins["xm"], ins["ym"])).sum()
    out["temperature"] = as_grid(grads(L, ins), ("DT", "tk2"))
    out["temperature"]["tkm"] = bar["rk4"]["tkm"]
    ins = {**leafs(["xm", "ym"], d), **leafs(["DSXX", "DSXY"], gr)}
    L = (dev["sxxm"] * P.interp("p", ins["DSXX"], ins["xm"], ins["ym"], lo=2, hi=1)).sum() \
        + (dev["sxym"] * P.interp("basic", ins["DSXY"], ins["xm"], ins["ym"])).sum()
    out["stress"] = as_grid(grads(L, ins), ("DSXX", "DSXY"))
    mi, gi = leafs(api.RK4_IN, d), leafs(api.RK4_GRIDS, gr)
    moved = P.rk4({**d, **mi}, gi, DT)
    q = grads(sum((dev[k] * moved[k]).sum() for k in dev), {**{"m_" + k: v for k, v in mi.items()},
                                                           **gi})
    out["rk4"] = {k: q["m_" + k].cpu().numpy() for k in mi}
    out["rk4_grids"] = as_grid({k: q[k] for k in gi}, api.RK4_GRIDS)
    return out
