"""Timed cases of the hydro advance: what a program that uses this package has
it do, from one small box to a 256^3 level, through the public Python entry
points over the C ABI.

Kinds of case (key "kind"):

* ``box``: the per-box drop-in of construct_hydro_source: hydro_ctoprim,
  hydro_srctoprim when there is a gravity source, hydro_umdrv, on the
  caller's device arrays.
* ``level``: steps of one level (computeNewDt + CAMR_advance), one box or
  many, Godunov PLM / PPM or the method of lines, periodic or with outflow
  and slip walls, with and without gravity, stepped or as captured graphs.
* ``refined``: steps of a refined level of uneven boxes over a sphere, its
  outer ghost cells from the coarser level.
* ``amr``: a subcycled step of a base level and a refined block of boxes
  (flux register, coarse-fine ghost fill, reflux, average down).
* ``eb``: a step of the Sod shock past a sphere with cut cells.
* ``adjoint``: the gradient of a density misfit after some steps.
* ``eb_adjoint``: the gradient of the force on the sphere.

All inputs are made from the seed: smooth random fields (8 density modes, a
k^-2 velocity spectrum at rms Mach 0.5, a smooth pressure, three species),
or Sod states whose pressures, densities and interface the seed moves.
Everything is float64.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from camr_amd import _lib, hydro, problems, workloads
from camr_amd.hydro import FluxRegister, Level, Problem

NV, NG = 10, 4
GAMMA = 1.4
RU, AIR_MW = 8.31446261815324e7, 26.93  # gas constant, molar mass of air (cgs)
PERIODIC, OUTFLOW, WALL = _lib.INTERIOR, _lib.OUTFLOW, _lib.SLIPWALL
MODEL_CFL = 0.4
MOL_CFL = 0.3  # the largest the method of lines takes
DEV = "cuda"

# Boundary sets: codes of the low and high faces per direction.
BCS = {
    "periodic": ((PERIODIC,) * 3, (PERIODIC,) * 3),
    "tube": ((OUTFLOW, PERIODIC, PERIODIC), (OUTFLOW, PERIODIC, PERIODIC)),
    "walls": ((OUTFLOW, WALL, WALL), (OUTFLOW, WALL, WALL)),
}


# ------------------------------------------------------------------ cases
def _box(nx, ny, nz, ppm, grav=0.0):
    return {"kind": "box", "nx": nx, "ny": ny, "nz": nz, "ppm": ppm, "grav": grav}


def _level(nx, ny, nz, ppm, bc="periodic", max_grid=0, grav=0.0, mol=0, graph=0, steps=1):
    return {"kind": "level", "nx": nx, "ny": ny, "nz": nz, "ppm": ppm, "bc": bc,
            "max_grid": max_grid, "grav": grav, "mol": mol, "graph": graph, "steps": steps}


def listed():
    return [
        # the smallest box of an adaptive hierarchy: latency and launches
        dict(_box(16, 16, 16, 0), name="box_plm_16"),
        # a clustered box with odd sides, PPM, with the gravity source term
        dict(_box(61, 37, 45, 1, -1.0), name="box_ppm_61x37x45_src"),
        # a box as large as hosts cut their grids
        dict(_box(128, 128, 128, 1), name="box_ppm_128"),
        # the shock tube that the reference ships as its first problem
        dict(_level(256, 4, 4, 0, "tube"), name="level_plm_sod_256x4x4"),
        # an odd level with outflow, walls and gravity
        dict(_level(97, 83, 61, 1, "walls", grav=-1.0), name="level_ppm_97x83x61_walls_grav"),
        # the refined level of a hierarchy: uneven boxes of 8 to 32 cells, as captured steps
        {"kind": "refined", "n": 128, "max_grid": 32, "graph": 1, "steps": 4, "name": "refined_ppm_128_sphere_graph"},
        # the headline level
        dict(_level(256, 256, 256, 1), name="level_ppm_256"),
        # the method of lines
        dict(_level(128, 128, 128, 0, mol=1), name="level_mol_128"),
        # two levels cut into boxes of at most 32, subcycled
        {"kind": "amr", "n": 96, "ppm": 1, "name": "amr_96_and_block"},
        # cut cells
        {"kind": "eb", "n": 64, "name": "eb_sod_sphere_128x64x64"},
        # gradients: a misfit after 10 steps, and the force on the sphere
        {"kind": "adjoint", "n": 96, "steps": 10, "every": 5, "name": "adjoint_ppm_96_10_steps"},
        {"kind": "eb_adjoint", "n": 32, "steps": 6, "every": 3, "name": "eb_adjoint_64x32x32_6_steps"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: sizes spread over their logarithm."""
    kind = rng.choice(("box", "box", "level", "level", "level", "refined", "amr", "eb", "adjoint", "eb_adjoint"))
    if kind == "box":
        n = [_log(rng, 8, 128) for _ in range(3)]
        return _box(*n, rng.randrange(2), rng.choice((0.0, 0.0, -1.0)))
    if kind == "level":
        form = rng.choice(("one", "one", "many", "mol", "tube"))
        if form == "tube":
            return _level(_log(rng, 64, 1024), rng.choice((4, 5, 8)), 4, rng.randrange(2), "tube")
        n = [_log(rng, 16, 160 if form == "one" else 128) for _ in range(3)]
        if form == "mol":
            return _level(*n, 0, rng.choice(("periodic", "walls")), mol=1)
        if form == "many":
            n = [max(x, 32) for x in n]
            return _level(*n, rng.randrange(2), max_grid=rng.choice((16, 32, 48)),
                          graph=rng.randrange(2), steps=rng.choice((1, 3)))
        return _level(*n, rng.randrange(2), rng.choice(("periodic", "walls")),
                      grav=rng.choice((0.0, 0.0, -1.0)))
    if kind == "refined":
        return {"kind": "refined", "n": 8 * rng.randrange(7, 17), "max_grid": rng.choice((16, 32, 64)),
                "graph": rng.randrange(2), "steps": rng.choice((1, 2))}
    if kind == "amr":
        return {"kind": "amr", "n": 8 * rng.randrange(4, 13), "ppm": rng.randrange(2)}
    if kind == "eb":
        return {"kind": "eb", "n": rng.randrange(28, 65)}
    if kind == "adjoint":
        return {"kind": "adjoint", "n": _log(rng, 24, 80), "steps": rng.randrange(4, 11), "every": rng.randrange(2, 6)}
    return {"kind": "eb_adjoint", "n": rng.randrange(20, 33), "steps": rng.randrange(4, 7), "every": rng.randrange(2, 4)}


# ----------------------------------------------------------------- inputs
def _field(n, seed, ghost=0):
    """Conserved state of the smooth random field at the cell centres of an
    (nx, ny, nz) periodic grid, grown by `ghost` cells that are no copies of
    the inside, as a device tensor (10, nz, ny, nx)."""
    r = np.random.default_rng(seed)
    m = [x + 2 * ghost for x in n]
    x, y, z = [(torch.arange(m[d], device=DEV, dtype=torch.float64) + 0.5) / m[d] for d in range(3)]
    x, y, z = x.view(1, 1, -1), y.view(1, -1, 1), z.view(-1, 1, 1)

    def modes(count, amp, kmax):
        f = torch.zeros(m[::-1], device=DEV, dtype=torch.float64)
        for _ in range(count):
            k = r.integers(-kmax, kmax + 1, size=3)
            f += amp * torch.sin(2 * math.pi * (int(k[0]) * x + int(k[1]) * y + int(k[2]) * z)
                                 + float(r.uniform(0, 2 * math.pi)))
        return f

    rho = 1.0 + modes(8, 0.1, 3)
    p = 1.0 + modes(3, 0.06, 2)
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    k = [torch.fft.fftfreq(m[d], 1.0 / m[d], device=DEV, dtype=torch.float64) for d in range(3)]
    kk = k[0].view(1, 1, -1) ** 2 + k[1].view(1, -1, 1) ** 2 + k[2].view(-1, 1, 1) ** 2
    filt = torch.where((kk >= 1) & (kk <= 256), 1.0 / kk.clamp(min=1.0), torch.zeros_like(kk))
    u = [torch.fft.ifftn(torch.fft.fftn(torch.randn(m[::-1], device=DEV, dtype=torch.float64, generator=g)) * filt).real
         for _ in range(3)]
    c2 = GAMMA * p / rho
    scale = 0.5 / math.sqrt(float(((u[0] ** 2 + u[1] ** 2 + u[2] ** 2) / c2).mean()))
    u = [scale * a for a in u]
    y0 = 0.5 + modes(2, 0.1, 2)
    y1 = 0.25 + modes(2, 0.05, 2)
    e = p / (GAMMA - 1.0)
    E = e + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return torch.stack([rho, rho * u[0], rho * u[1], rho * u[2], E, e, torch.zeros_like(rho),
                        rho * y0, rho * y1, rho * (1.0 - y0 - y1)])


def _sod(lo, hi, dx, seed, interface):
    """Sod states whose left and right pressure and density and whose
    interface the seed moves by up to a tenth."""
    r = np.random.default_rng(seed)
    a = [float(v) for v in r.uniform(0.9, 1.1, size=5)]
    return problems.sod(lo, hi, dx, p_l=a[0], p_r=0.1 * a[1], rho_l=a[2], rho_r=0.125 * a[3],
                        interface=interface * a[4])


class _BoxMemory:
    """A box of a level as torch takes foreign memory.  The tensor made of it
    holds this object, and so the level, whose memory ends with it."""

    def __init__(self, level, b):
        self.level = level
        self.__cuda_array_interface__ = {"shape": level.shape(b), "typestr": "<f8",
                                         "data": (level.state_array(b).p, False), "version": 3}


def _state(level):
    """The level's new-time state as device tensors, one per box (a view of
    the level's own memory)."""
    return [torch.as_tensor(_BoxMemory(level, b), device=DEV) for b in range(len(level.boxes))]


class _Views:
    """State views of a level, kept for each of its two time buffers."""

    def __init__(self, level):
        self.level, self.kept = level, {}

    def __call__(self):
        key = self.level.state_array(0).p
        if key not in self.kept:
            self.kept[key] = _state(self.level)
        return self.kept[key]


def _coarsened(U):
    n = U.shape[1] // 2
    return U.view(NV, n, 2, n, 2, n, 2).mean(dim=(2, 4, 6))


def _chop(n, mg):
    mg = mg or max(n)
    return [(i, j, k, min(i + mg, n[0]) - 1, min(j + mg, n[1]) - 1, min(k + mg, n[2]) - 1)
            for k in range(0, n[2], mg) for j in range(0, n[1], mg) for i in range(0, n[0], mg)]


def _put(level, U):
    """The level's boxes from the global field U, then initData's tail."""
    for v, b in zip(_state(level), level.boxes):
        v.copy_(U[:, b[2]:b[5] + 1, b[1]:b[4] + 1, b[0]:b[3] + 1])
    level.init_post()


def _sizes(c):
    return [c["nx"], c["ny"], c["nz"]]


def _level_input(c, seed):
    n = _sizes(c)
    if c["bc"] == "tube":
        return torch.as_tensor(_sod((0, 0, 0), [x - 1 for x in n], (1.0 / n[0],) * 3, seed, 0.5), device=DEV)
    return _field(n, seed)


def _level_problem(c):
    n = _sizes(c)
    bclo, bchi = BCS[c["bc"]]
    return Problem(domlo=(0, 0, 0), domhi=tuple(x - 1 for x in n), dx=(1.0 / max(n),) * 3, bclo=bclo, bchi=bchi,
                   is_periodic=tuple(int(b == PERIODIC) for b in bclo), boxes=_chop(n, c["max_grid"]),
                   params=dict(ppm_type=c["ppm"], do_mol=c["mol"], const_grav=c["grav"],
                               cfl=MOL_CFL if c["mol"] else MODEL_CFL))


def _box_problem(c):
    n = _sizes(c)
    return Problem(domlo=(-1000,) * 3, domhi=(1000,) * 3, dx=(1.0 / max(n),) * 3, bclo=(PERIODIC,) * 3,
                   bchi=(PERIODIC,) * 3, is_periodic=(1, 1, 1), boxes=[(0, 0, 0) + tuple(x - 1 for x in n)],
                   params=dict(ppm_type=c["ppm"]))


def _box_dt(c):
    return 0.1 / max(_sizes(c))


@functools.lru_cache(maxsize=8)
def _refined(n, max_grid):
    return workloads.refined_level(n=n, max_size=max_grid, ppm_type=1, cfl=MODEL_CFL)


def _block(n, ppm):
    """The refined level of an amr case: the middle half of the domain of the
    doubled resolution, in boxes of at most 32 aligned to it."""
    lo, hi = 2 * (n // 4), 2 * (n - n // 4)
    boxes = [tuple(lo + x for x in b) for b in _chop([hi - lo] * 3, 32)]
    return Problem(domlo=(0, 0, 0), domhi=(2 * n - 1,) * 3, dx=(0.5 / n,) * 3, bclo=(PERIODIC,) * 3,
                   bchi=(PERIODIC,) * 3, is_periodic=(1, 1, 1), boxes=boxes,
                   params=dict(ppm_type=ppm, cfl=MODEL_CFL))


@functools.lru_cache(maxsize=8)
def _sphere(n):
    prob = workloads.sod_sphere(n=n, max_grid=32, cfl=0.3)
    return prob, workloads.sod_sphere_geometry(prob)


def _eb_level(n, seed, smooth):
    prob, geom = _sphere(n)
    level = Level(prob, engine=_lib.ENGINE_STAGED)
    level.set_eb(geom)
    amp = float(np.random.default_rng(seed).uniform(0.15, 0.25))
    for b, v in enumerate(_state(level)):
        lo, hi = prob.boxes[b][:3], prob.boxes[b][3:]
        if smooth:
            U = workloads.sod_sphere_smooth_init(prob, b, geom, amp=amp)
        else:
            U = _sod(lo, hi, prob.dx, seed, prob.interface)
            U[:, geom.covered_mask(lo, hi)] = 0.0
        v.copy_(torch.as_tensor(U))
    level.init_post()
    return level


def _adjoint_field(n, seed):
    """The smooth field with one species, as the misfit's tests take it."""
    U = _field([n] * 3, seed)
    U[7], U[8:] = U[0], 0.0
    return U


def _adjoint_problem(n):
    return workloads.smooth_periodic(n=n, ppm_type=1, cfl=MODEL_CFL)


def _adjoint_dts(c):
    # a fixed sequence below the CFL limit of every seed's field
    return np.full(c["steps"], 0.08 / c["n"])


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "box":
        n = _sizes(c)
        prob = _box_problem(c)
        U = _field(n, seed, NG)
        new = lambda nc, g=NG, d=-1: torch.empty(  # noqa: E731
            (nc,) + tuple(n[a] + 2 * g + (a == d) for a in (2, 1, 0)), device=DEV, dtype=torch.float64)
        s = {"kind": kind, "U": U, "q": new(11), "qa": new(5), "params": hydro.hydro_params(prob),
             "lo": (0, 0, 0), "hi": tuple(x - 1 for x in n), "dt": _box_dt(c),
             "dsdt": new(NV, 0), "flx": [new(NV, 0, d) for d in range(3)], "src": None, "srcq": None}
        if c["grav"]:
            s["src"] = torch.zeros_like(U)
            s["src"][3], s["src"][4] = c["grav"] * U[0], c["grav"] * U[3]
            s["srcq"] = new(11)
        return s
    if kind == "level":
        level = Level(_level_problem(c), graph=bool(c["graph"]))
        _put(level, _level_input(c, seed))
        return {"kind": kind, "level": level, "view": _Views(level), "dt": level.initial_dt(),
                "steps": c["steps"], "graph": c["graph"]}
    if kind == "refined":
        n = c["n"]
        coarse = Level(workloads.smooth_periodic(n=n // 2, ppm_type=1, cfl=MODEL_CFL, max_grid=32))
        level = Level(_refined(n, c["max_grid"]), graph=bool(c["graph"]))
        U = _field([n] * 3, seed)
        _put(level, U)
        _put(coarse, _coarsened(U))
        level.exterior_from_coarse(coarse, 2)
        return {"kind": kind, "level": level, "view": _Views(level), "dt": level.initial_dt(), "coarse": coarse,
                "steps": c["steps"], "graph": c["graph"]}
    if kind == "amr":
        n = c["n"]
        coarse = Level(workloads.smooth_periodic(n=n, ppm_type=c["ppm"], cfl=MODEL_CFL, max_grid=32))
        fine = Level(_block(n, c["ppm"]))
        reg = FluxRegister(coarse, fine, 2)
        U = _field([2 * n] * 3, seed)
        _put(fine, U)
        _put(coarse, _coarsened(U))
        coarse.average_down(fine, 2)
        coarse.init_post()
        return {"kind": kind, "reg": reg, "coarse": coarse, "fine": fine, "views": (_Views(coarse), _Views(fine)),
                "dt": min(coarse.initial_dt(), 2 * fine.initial_dt())}
    if kind == "eb":
        level = _eb_level(c["n"], seed, False)
        return {"kind": kind, "level": level, "view": _Views(level), "dt": level.initial_dt(), "steps": 1, "graph": 0}
    if kind == "adjoint":
        level = Level(_adjoint_problem(c["n"]))
        _put(level, _adjoint_field(c["n"], seed))
        return {"kind": kind, "level": level, "dts": _adjoint_dts(c), "every": c["every"],
                "target": _adjoint_field(c["n"], seed + 1)[0].cpu().numpy()}
    level = _eb_level(c["n"], seed, True)
    return {"kind": kind, "level": level, "dts": np.full(c["steps"], 0.1 / c["n"]), "every": c["every"]}


# -------------------------------------------------------------- one pass
def _whole(boxes):
    """The state of a few boxes as it is, of many as one tensor."""
    return boxes if len(boxes) <= 40 else [torch.cat([b.reshape(-1) for b in boxes])]


def run(state):
    s, kind = state, state["kind"]
    if kind == "box":
        g = [-NG] * 3
        gh = [h + NG for h in s["hi"]]
        s["dsdt"].zero_()
        hydro.hydro_ctoprim(g, gh, s["U"], g, s["q"], s["qa"], s["params"])
        if s["src"] is not None:
            hydro.hydro_srctoprim(g, gh, s["q"], s["qa"], s["src"], s["srcq"])
        hydro.hydro_umdrv(s["lo"], s["hi"], s["U"], g, s["dsdt"], s["q"], s["qa"], s["srcq"], s["flx"], s["dt"],
                          s["params"])
        return {"dsdt": s["dsdt"], "flx": s["flx"]}
    if kind in ("level", "refined", "eb"):
        if kind == "refined":
            s["level"].exterior_from_coarse(s["coarse"], 2)
        if s["graph"] or s["steps"] > 1:
            dts = s["level"].run(s["steps"])
        else:
            s["dt"] = s["level"].new_dt(s["dt"])
            s["level"].advance(s["dt"])
            dts = s["dt"]
        return {"dt": dts, "state": _whole(s["view"]())}
    if kind == "amr":
        C, F = s["coarse"], s["fine"]
        s["dt"] = min(C.new_dt(s["dt"]), 2 * F.new_dt(s["dt"] / 2))
        hydro.amr_step(C, F, s["reg"], s["dt"])
        return {"dt": s["dt"], "coarse": _whole(s["views"][0]()), "fine": _whole(s["views"][1]())}
    level = s["level"]
    level.adjoint_forward(s["dts"], s["every"])
    if kind == "adjoint":
        seed = np.zeros(level.shape(0))
        rho = level.get_box(0)[0]
        seed[0] = rho - s["target"]
        level.set_adjoint(0, seed)
    else:
        level.seed_force_adjoint((1.0, 0.0, 0.0))
    level.adjoint_backward()
    grad = [level.get_adjoint(b) for b in range(len(level.boxes))]
    return {"rho": rho, "grad": grad} if kind == "adjoint" else {"grad": grad}


# ------------------------------------------------------------------ work
# FP64 operations of one cell-update of the reference's algorithm (additions,
# multiplications, divisions, square roots, one each), counted at 256^3
# (PPM) and from its share of the traces at 32^3 (PLM); the method of lines
# has two stages without transverse solves.
FLOP = {"ppm": 6576.0, "plm": 4640.0, "mol": 2400.0}


def _cells(boxes):
    return sum((b[3] - b[0] + 1) * (b[4] - b[1] + 1) * (b[5] - b[2] + 1) for b in boxes)


def work(case):
    """State read once and written once per pass (the grown box, fluxes and
    dS/dt for a box), and the algorithm's operations."""
    c, kind = case, case["kind"]
    if kind == "box":
        n = _sizes(c)
        cells, grown = np.prod([float(x) for x in n]), np.prod([float(x + 2 * NG) for x in n])
        faces = sum(cells / x * (x + 1) for x in n)
        per = FLOP["ppm" if c["ppm"] else "plm"]
        return {"bytes": 8 * (grown * (NV * (2 if c["grav"] else 1) + 16 + (11 if c["grav"] else 0))
                              + NV * (faces + cells)), "flops": per * cells}
    if kind == "level":
        cells = float(np.prod([float(x) for x in _sizes(c)]))
        per = FLOP["mol"] if c["mol"] else FLOP["ppm" if c["ppm"] else "plm"]
        return {"bytes": 16 * NV * cells, "flops": per * cells * c["steps"]}
    if kind == "refined":
        cells = _cells(_refined(c["n"], c["max_grid"]).boxes)
        return {"bytes": 16.0 * NV * cells, "flops": FLOP["ppm"] * cells * c["steps"]}
    if kind == "amr":
        n = c["n"]
        fine = _cells(_block(n, c["ppm"]).boxes)
        return {"bytes": 16.0 * NV * (n ** 3 + fine),
                "flops": FLOP["ppm" if c["ppm"] else "plm"] * float(n ** 3 + 2 * fine)}
    cells = 2.0 * c["n"] ** 3 if kind.startswith("eb") else float(c["n"] ** 3)
    if kind == "eb":
        return {"bytes": 16 * NV * cells, "flops": FLOP["plm"] * cells}
    # each step forward, recomputed, and in reverse at about two forward steps
    per = FLOP["ppm" if kind == "adjoint" else "plm"]
    return {"bytes": 8.0 * NV * cells * (c["steps"] + 2), "flops": 4 * per * cells * c["steps"]}


def tolerance(case):
    """The forward paths promise the reference's bits: every operation of the
    reference, rounded as there.  The gradients are sums whose order is the
    implementation's: the same inputs twice differ by up to 2e-16 of the norm
    and 8e-15 in one entry, a plain restatement by 7e-16 of the norm."""
    if case["kind"] in ("adjoint", "eb_adjoint"):
        return {"rel": 3e-15, "max": 1e-12}
    return "exact"


# ----------------------------------------------- a plain torch restatement
# One step of the single-level path in plain float64 tensor operations: state
# arrays (component, z, y, x) with NG ghost cells, neighbours by rolling.
SMALL, SMALL_DENS, SMALL_PRES, SMALLU, DIFMAG = 1e-8, 1e-7, 1e-200, 1e-12, 0.1


def _sh(x, d, o=1):
    return torch.roll(x, -o, dims=x.dim() - 1 - d)


def _edge(x, d, at):
    """Index of position `at` along direction d of the last three axes."""
    i = [slice(None)] * x.dim()
    i[x.dim() - 1 - d] = at
    return tuple(i)


def _ghosts(U, bc):
    """FillPatch of a one-box level: periodic, outflow (copied edge), walls."""
    for d in range(3):
        n = U.shape[3 - d]
        i = torch.arange(-NG, n + NG, device=U.device)
        lo, hi = i < 0, i >= n
        src, flip = i.clone(), torch.ones(n + 2 * NG, device=U.device, dtype=U.dtype)
        for side, code in ((lo, bc[0][d]), (hi, bc[1][d])):
            if code == PERIODIC:
                src = torch.where(side, i % n, src)
            elif code == WALL:
                src = torch.where(side, torch.where(i < 0, -i - 1, 2 * n - 1 - i), src)
                flip = torch.where(side, -flip, flip)
            else:
                src = torch.where(side, i.clamp(0, n - 1), src)
        U = U.index_select(3 - d, src)
        sign = torch.ones((NV,) + tuple(n + 2 * NG if a == d else 1 for a in (2, 1, 0)), device=U.device, dtype=U.dtype)
        sign[1 + d] = flip.view(sign.shape[1:])
        U = U * sign
    return U


def _clean(U):
    rho = U[0]
    ke = 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / rho
    e = U[4] - ke
    take = (e > 0) & (e / U[4] > 1e-4)
    eint = torch.where(take, e, U[5])
    E = torch.where(take, U[4], eint + ke)
    y = torch.minimum(U[7:], rho).clamp(min=0.0)
    y = y / (y.sum(0) / rho)
    T = (GAMMA - 1.0) * eint / rho * AIR_MW / RU
    return torch.cat([torch.stack([rho, U[1], U[2], U[3], E, eint, T]), y])


def _prim(U):
    """rho, u, v, w, p, rho e, Y0..Y2 and the sound speed."""
    r = U[0]
    p = (GAMMA - 1.0) * U[5]
    return torch.cat([torch.stack([r, U[1] / r, U[2] / r, U[3] / r, p, U[5]]), U[7:] / r]), torch.sqrt(GAMMA * p / r)


def _flat(q):
    f = torch.ones_like(q[4])
    for d in range(3):
        P = {o: _sh(q[4], d, o) for o in range(-3, 4)}
        V = {o: _sh(q[1 + d], d, o) for o in range(-2, 3)}

        def at(s):
            dp = P[s + 1] - P[s - 1]
            zeta = dp.abs() / (P[s + 2] - P[s - 2]).abs().clamp(min=1e-200)
            z = ((zeta - 0.75) / 0.1).clamp(0.0, 1.0)
            on = (V[s - 1] - V[s + 1] >= 0) & (dp.abs() / torch.minimum(P[s + 1], P[s - 1]) > 0.33)
            return torch.where(on, z, torch.zeros_like(z))
        fd = 1.0 - torch.maximum(at(0), torch.where(P[1] - P[-1] > 0, at(-1), at(1)))
        n = fd.shape[2 - d]
        for i in (0, 1, 2, n - 3, n - 2, n - 1):
            m = torch.zeros(n, device=fd.device, dtype=torch.bool)
            m[i] = True
            fd = torch.where(m.view([n if a == d else 1 for a in (2, 1, 0)]), torch.ones_like(fd), fd)
        f = torch.minimum(f, fd)
    return f


def _mc(a, b, c):
    """Van Leer's limited difference of the triple."""
    l, r = b - a, c - b
    m = torch.minimum(0.5 * (l + r).abs(), 2.0 * torch.minimum(l.abs(), r.abs()))
    return torch.where(l * r > 0, torch.copysign(m, l + r), torch.zeros_like(m))


def _others(d):
    return [t for t in range(3) if t != d]


def _ppm(q, c, fl, d, dtdx):
    un = q[1 + d]
    Ip, Im = [], []
    for s in range(9):
        a = [_sh(q[s], d, o) for o in range(-2, 3)]
        dl, dc, dr = _mc(a[0], a[1], a[2]), _mc(a[1], a[2], a[3]), _mc(a[2], a[3], a[4])

        def edge(x, y, dx, dy):
            e = 0.5 * (y + x) - (dy - dx) / 6.0
            return torch.minimum(torch.maximum(e, torch.minimum(x, y)), torch.maximum(x, y))
        sm, sp = edge(a[1], a[2], dl, dc), edge(a[2], a[3], dc, dr)
        sm, sp = fl * sm + (1 - fl) * a[2], fl * sp + (1 - fl) * a[2]
        ext = (sp - a[2]) * (a[2] - sm) <= 0
        big = (sp - a[2]).abs() >= 2 * (sm - a[2]).abs()
        low = ~big & ((sm - a[2]).abs() >= 2 * (sp - a[2]).abs())
        sp, sm = (torch.where(ext, a[2], torch.where(big, 3 * a[2] - 2 * sm, sp)),
                  torch.where(ext, a[2], torch.where(low, 3 * a[2] - 2 * sp, sm)))
        s6 = 6 * a[2] - 3 * (sm + sp)
        ip, im = [], []
        for w, v in enumerate((un - c, un, un + c)):
            if 4 > s != 1 + d and s > 0 or s > 5:  # passive: the contact wave only
                if w != 1:
                    ip.append(None)
                    im.append(None)
                    continue
            sg = v.abs() * dtdx
            k = (1 - (2.0 / 3.0) * sg) * s6
            ip.append(torch.where(v <= 0, sp, sp - 0.5 * sg * (sp - sm - k)))
            im.append(torch.where(v <= 0, sm + 0.5 * sg * (sp - sm + k), sm))
        Ip.append(ip)
        Im.append(im)

    def project(I, plus):
        w = 0 if plus else 2
        rho, p = I[0][w].clamp(min=SMALL_DENS), I[4][w].clamp(min=SMALL_PRES)
        u, re = I[1 + d][w], I[5][w]
        cr = torch.sqrt(GAMMA * p / rho)
        h = (p + re) / rho / cr ** 2
        am = 0.5 * ((p - I[4][0]) / (rho * cr) - (u - I[1 + d][0])) * rho / cr
        ap = 0.5 * ((p - I[4][2]) / (rho * cr) + (u - I[1 + d][2])) * rho / cr
        ar = rho - I[0][1] - (p - I[4][1]) / cr ** 2
        ae = re - I[5][1] - (p - I[4][1]) * h

        def use(v):  # the wave's part that reaches this face
            on = v < 0 if plus else v > 0
            return torch.where(on, -torch.ones_like(v), torch.where(v == 0, -0.5 * torch.ones_like(v), torch.zeros_like(v)))
        am, ap, f0 = am * use(un - c), ap * use(un + c), use(un)
        o = [None] * 9
        o[0] = (rho + ap + am + ar * f0).clamp(min=SMALL_DENS)
        o[1 + d] = u + (ap - am) * cr / rho
        o[4] = (p + (ap + am) * cr ** 2).clamp(min=SMALL_PRES if plus else SMALL_DENS)
        o[5] = re + (ap + am) * h * cr ** 2 + ae * f0
        for s in [1 + t for t in _others(d)] + [6, 7, 8]:
            o[s] = I[s][1]
        return torch.stack(o)
    return project(Im, True), _sh(project(Ip, False), d, -1)


def _plm(q, c, fl, d, dtdx):
    sl = []
    for s in range(9):
        a = [_sh(q[s], d, o) for o in range(-2, 3)]
        l, r = a[2] - a[1], a[3] - a[2]
        lim = torch.where(l * r >= 0, 2 * torch.minimum(l.abs(), r.abs()), torch.zeros_like(l))
        cen = 0.5 * (l + r)
        t = 4.0 / 3.0 * cen - (_mc(a[2], a[3], a[4]) + _mc(a[0], a[1], a[2])) / 6.0
        sl.append(fl * torch.copysign(torch.minimum(lim, t.abs()), cen))
    rho, p, re, un = q[0], q[4], q[5], q[1 + d]
    t1, t2 = [1 + t for t in _others(d)]
    cs = c * c
    h = (re + p) / rho / cs
    am = 0.5 * (sl[4] / (rho * c) - sl[1 + d]) * rho / c
    ap = 0.5 * (sl[4] / (rho * c) + sl[1 + d]) * rho / c
    a0 = {0: sl[0] - sl[4] / cs, 5: sl[5] - sl[4] * h, t1: sl[t1], t2: sl[t2]}
    out = []
    for sgn in (-1, 1):
        ref, far = (un - c, un + c) if sgn < 0 else (un + c, un - c)
        fac = 0.5 * (sgn - dtdx * (ref.clamp(max=0) if sgn < 0 else ref.clamp(min=0)))
        on = lambda v: 1 + sgn * torch.copysign(torch.ones_like(v), v)  # noqa: E731
        acoustic = 0.25 * dtdx * (ref - far) * on(far) * (ap if sgn < 0 else am)
        z = 0.25 * dtdx * (ref - un) * on(un)
        o = [None] * 9
        o[0] = (rho + fac * sl[0] + acoustic + z * a0[0]).clamp(min=SMALL_DENS)
        o[1 + d] = un + fac * sl[1 + d] - sgn * acoustic * c / rho
        o[t1], o[t2] = q[t1] + fac * sl[t1] + z * a0[t1], q[t2] + fac * sl[t2] + z * a0[t2]
        o[4] = (p + fac * sl[4] + acoustic * cs).clamp(min=SMALL_PRES)
        o[5] = re + fac * sl[5] + acoustic * h * cs + z * a0[5]
        v = torch.where(un > 0, -torch.ones_like(un), un * dtdx) if sgn < 0 else torch.where(un >= 0, un * dtdx, torch.ones_like(un))
        for s in (6, 7, 8):
            o[s] = q[s] + 0.5 * (sgn - v) * sl[s]
        out.append(torch.stack(o))
    return out[0], _sh(out[1], d, -1)


def _riemann(ql, qr, c, d, bc):
    """Fluxes rho, mx, my, mz, E, e, Y0..Y2 and the face's u and p; the states
    at walls and outflow faces are the inside's."""
    for side in (0, 1):
        code = bc[side][d]
        if code == PERIODIC:
            continue
        at = _edge(ql, d, NG if side == 0 else ql.shape[3 - d] - NG)
        ins, out = (qr, ql) if side == 0 else (ql, qr)
        out = out.clone()
        v, y = ins[at].clone(), out[at][6:].clone()
        if code == WALL:
            v[1 + d] = -v[1 + d]
        out[at] = torch.cat([v[:6], y])
        ql, qr = (out, qr) if side == 0 else (ql, out)
    cl = _sh(c, d, -1)
    cav, smallc = 0.5 * (c + cl), SMALL * torch.maximum(torch.maximum(c, cl), torch.ones_like(c))
    rl, rr = ql[0].clamp(min=SMALL_DENS), qr[0].clamp(min=SMALL_DENS)
    pl, pr = ql[4].clamp(min=SMALL_PRES), qr[4].clamp(min=SMALL_PRES)
    ul, ur = ql[1 + d], qr[1 + d]
    wl = torch.maximum(smallc * SMALL_DENS, torch.sqrt((GAMMA * pl * rl).abs()))
    wr = torch.maximum(smallc * SMALL_DENS, torch.sqrt((GAMMA * pr * rr).abs()))
    ps = ((wr * pl + wl * pr + wl * wr * (ul - ur)) / (wl + wr)).clamp(min=SMALL_PRES)
    us = (wl * ul + wr * ur + (pl - pr)) / (wl + wr)
    us = torch.where(us.abs() < SMALLU * 0.5 * (ul.abs() + ur.abs()), torch.zeros_like(us), us)
    pick = lambda a, b: torch.where(us > 0, a, torch.where(us < 0, b, 0.5 * (a + b)))  # noqa: E731
    ro, uo, po, eo = pick(rl, rr).clamp(min=SMALL_DENS), pick(ul, ur), pick(pl, pr), pick(ql[5], qr[5])
    co = torch.maximum(smallc, torch.sqrt((GAMMA * po / ro).abs()))
    dp = ps - po
    rs = (ro + dp / co ** 2).clamp(min=SMALL_DENS)
    es = eo + dp * (eo + po) / ro / co ** 2
    cs = torch.maximum(torch.sqrt((GAMMA * ps / rs).abs()), smallc)
    sg = torch.where(us < 0, -1.0, 1.0).to(us.dtype)
    out, inn = co - sg * uo, cs - sg * us
    shock = 0.5 * (inn + out)
    out, inn = torch.where(dp > 0, shock, out), torch.where(dp > 0, shock, inn)
    df = out - inn
    fr = (0.5 * (1 + (out + inn) / torch.where(df == 0, SMALL * cav, df))).clamp(0.0, 1.0)

    def fan(star, o):
        v = torch.where(out < 0, o, fr * star + (1 - fr) * o)
        return torch.where(inn >= 0, star, v)
    rho, un, p, re = fan(rs, ro), fan(us, uo), fan(ps, po).clamp(min=SMALL_PRES), fan(es, eo)
    vel = [un if t == d else pick(ql[1 + t], qr[1 + t]) for t in range(3)]
    fr_ = rho * un
    E = re + 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    f = [fr_] + [fr_ * v + (p if t == d else 0.0) for t, v in enumerate(vel)] + [un * (E + p), un * re]
    f += [fr_ * pick(ql[6 + s], qr[6 + s]) for s in range(3)]
    return torch.stack(f), un, p, ql, qr


def _corrected(q, D, pcorr, src=None):
    """A face state after its conserved part loses D and its pressure pcorr."""
    r = q[0]
    n = [r * q[1 + t] - D[1 + t] for t in range(3)]
    E = q[5] + 0.5 * r * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) - D[4]
    rn = r - D[0]
    o = [rn] + [x / rn for x in n] + [(q[4] - pcorr), E - 0.5 * (n[0] ** 2 + n[1] ** 2 + n[2] ** 2) / rn]
    o += [(r * q[6 + s] - D[6 + s]) / rn for s in range(3)]
    if src is not None:
        o[3] = o[3] + src
    o[4] = o[4].clamp(min=SMALL_PRES)
    return torch.stack(o)


def _work(p, u, t):
    """d(p u) + (gamma - 1) <p> du across the cell in direction t."""
    pr, ur = _sh(p, t), _sh(u, t)
    return pr * ur - p * u + 0.5 * (pr + p) * (ur - u) * (GAMMA - 1.0)


def _divu(q, dx):
    def mean(v, a, b):
        v = v + _sh(v, a, -1)
        return 0.25 * (v + _sh(v, b, -1))
    return sum(mean(q[1 + d] - _sh(q[1 + d], d, -1), *_others(d)) / dx for d in range(3))


def _finish(f, u, U, div, d, dx):
    """Artificial viscosity, species normalisation, area: the NV fluxes."""
    t = _others(d)
    a = div + _sh(div, t[0])
    v = dx * DIFMAG * (0.25 * (a + _sh(a, t[1]))).clamp(max=0.0)
    F = [f[n] + v * (U[n] - _sh(U[n], d, -1)) for n in range(6)]
    Y = [f[6 + s] + v * (U[7 + s] - _sh(U[7 + s], d, -1)) for s in range(3)]
    s = Y[0] + Y[1] + Y[2]
    fac = torch.where(s != 0, F[0] / s, torch.ones_like(s))
    return torch.stack(F + [torch.zeros_like(s)] + [y * fac for y in Y]) * dx * dx


def _godunov(U, dt, dx, ppm, bc, srcw=None):
    """Final fluxes (area included) and face (u, p) on the grown arrays."""
    q, c = _prim(U)
    fl = _flat(q)
    qp, qm, F1 = [], [], []
    for d in range(3):
        a, b = (_ppm if ppm else _plm)(q, c, fl, d, dt / dx)
        f, u, p, b, a = _riemann(b, a, c, d, bc)
        qp.append(a)
        qm.append(b)
        F1.append((f, u, p))
    F2 = {}
    for t in range(3):
        f, u, p = F1[t]
        k = dt / (3 * dx)
        D, w = k * (_sh(f, t) - f), k * _work(p, u, t)
        for d in _others(t):
            F2[d, t] = _riemann(_corrected(qm[d], _sh(D, d, -1), _sh(w, d, -1)), _corrected(qp[d], D, w), c, d, bc)[:3]
    div = _divu(q, dx)
    out = []
    for d in range(3):
        a, b = _others(d)
        k = 0.5 * dt / dx
        (fa, ua, pa), (fb, ub, pb) = F2[a, b], F2[b, a]
        D = k * (_sh(fa, a) - fa + _sh(fb, b) - fb)
        w = k * (_work(pa, ua, a) + _work(pb, ub, b))
        s = None if srcw is None else 0.5 * dt * srcw
        f, u, p = _riemann(_corrected(qm[d], _sh(D, d, -1), _sh(w, d, -1), None if s is None else _sh(s, d, -1)),
                           _corrected(qp[d], D, w, s), c, d, bc)[:3]
        out.append((_finish(f, u, U, div, d, dx), u, p))
    return out


def _mol_fluxes(U, dx, bc):
    q, c = _prim(U)
    div = _divu(q, dx)
    out = []
    for d in range(3):
        t1, t2 = [1 + t for t in _others(d)]
        h = (q[5] + q[4]) / q[0]
        up, dn = _sh(q, d, 1), _sh(q, d, -1)

        def waves(b, a):  # differences of the characteristic variables b - a
            dp, du = b[4] - a[4], b[1 + d] - a[1 + d]
            w = [0.5 * dp / c - 0.5 * q[0] * du, 0.5 * dp / c + 0.5 * q[0] * du, b[t1] - a[t1], b[t2] - a[t2],
                 b[5] - a[5] - h * dp / c ** 2]
            return w + [b[0] * b[s] - a[0] * a[s] - q[s] * dp / c ** 2 for s in (6, 7, 8)]
        dq = []
        for l, r in zip(waves(q, dn), waves(up, q)):
            cen = 0.5 * (l + r)
            lim = torch.where(l * r >= 0, 2 * torch.minimum(l.abs(), r.abs()), torch.zeros_like(l))
            dq.append(torch.copysign(torch.minimum(lim, cen.abs()), cen))
        ac = dq[0] + dq[1]
        st = []
        for s in (-0.5, 0.5):
            o = [None] * 9
            o[4] = (q[4] + s * ac * c).clamp(min=SMALL_PRES)
            o[1 + d] = q[1 + d] + s * (dq[1] - dq[0]) / q[0]
            o[t1], o[t2] = q[t1] + s * dq[2], q[t2] + s * dq[3]
            y = [q[0] * q[6 + n] + s * (dq[5 + n] + q[6 + n] * ac / c) for n in range(3)]
            tot = y[0] + y[1] + y[2]
            o[0] = tot.clamp(min=SMALL_DENS)
            o[6:] = [v / tot for v in y]
            o[5] = q[5] + s * (dq[4] + h * ac / c)
            st.append(torch.stack(o))
        f, u, p = _riemann(_sh(st[1], d, -1), st[0], c, d, bc)[:3]
        out.append((_finish(f, u, U, div, d, dx), u, p))
    return out


def _dsdt(F, dx):
    vol, area = dx ** 3, dx * dx
    ds = sum(f - _sh(f, d) for d, (f, u, p) in enumerate(F)) / vol
    pd = 0.5 * sum((_sh(p, d) + p) * (_sh(u, d) - u) * area for d, (f, u, p) in enumerate(F)) / vol
    e = torch.zeros(NV, 1, 1, 1, device=ds.device, dtype=ds.dtype)
    e[5] = 1.0
    return ds - e * pd


def _inner(x):
    return x[..., NG:-NG, NG:-NG, NG:-NG]


def _step(S, dt, dx, c, bc):
    """One step of a level that is one box (or whose boxes see no shock)."""
    S = _clean(S)
    U = _clean(_ghosts(S, bc))
    g = c.get("grav", 0.0)
    if c.get("mol"):
        S1 = _inner(U) + dt * _inner(_dsdt(_mol_fluxes(U, dx, bc), dx))
        U = _clean(_ghosts(S1, bc))
        new = 0.5 * _inner(U) + 0.5 * S + 0.5 * dt * _inner(_dsdt(_mol_fluxes(U, dx, bc), dx))
        return _clean(_clean(new))
    srcw = None
    if g:  # the source's velocity part: g inside and in periodic ghosts
        srcw = torch.full_like(S[0], g)
        for d in range(3):
            if bc[0][d] == PERIODIC:
                srcw = torch.cat([srcw.narrow(2 - d, 0, NG), srcw, srcw.narrow(2 - d, 0, NG)], 2 - d)
            else:
                z = torch.zeros_like(srcw.narrow(2 - d, 0, NG))
                srcw = torch.cat([z, srcw, z], 2 - d)
    new = _inner(U) + dt * _inner(_dsdt(_godunov(U, dt, dx, c["ppm"], bc, srcw), dx))
    if g:
        new = new + dt * g * _mom(S[0], S[3])
    new = _clean(new)
    if g:
        new = _clean(new + 0.5 * dt * g * _mom(new[0] - S[0], new[3] - S[3]))
    return _clean(new)


def _mom(w, e):
    z = torch.zeros_like(w)
    return torch.stack([z, z, z, w, e, z, z, z, z, z])


def _cfl_dt(S, dx, cfl):
    c = torch.sqrt(GAMMA * (GAMMA - 1.0) * S[5] / S[0])
    return cfl * float(min((dx / (c + (S[1 + d] / S[0]).abs())).min() for d in range(3)))


def exact(case, seed):
    """run()'s outputs from the restatement; None for the coarse-fine and
    cut-cell kinds, whose plain restatement is beyond this file, and for
    gradients too long to differentiate in a few seconds."""
    c, kind = case, case["kind"]
    if kind == "box":
        n = _sizes(c)
        U, dx = _field(n, seed, NG), 1.0 / max(n)
        srcw = torch.full_like(U[0], c["grav"]) if c["grav"] else None
        F = _godunov(U, _box_dt(c), dx, c["ppm"], BCS["periodic"], srcw)
        flx = []
        for d in range(3):
            f = F[d][0]
            for a in range(3):
                f = f.narrow(3 - a, NG, n[a] + (a == d))
            flx.append(f)
        return {"dsdt": _inner(_dsdt(F, dx)), "flx": flx}
    if kind == "level":
        n = _sizes(c)
        prob = _level_problem(c)
        bc, dx = BCS[c["bc"]], prob.dx[0]
        S = _clean(_level_input(c, seed))
        dts = []
        for _ in range(c["steps"]):
            dt = _cfl_dt(S, dx, prob.params["cfl"])
            dts.append(min(dt, 1.1 * dts[-1]) if dts else dt)
            S = _step(S, dts[-1], dx, c, bc)
        boxes = [S[:, b[2]:b[5] + 1, b[1]:b[4] + 1, b[0]:b[3] + 1] for b in prob.boxes]
        return {"dt": np.array(dts) if c["graph"] or c["steps"] > 1 else dts[0], "state": _whole(boxes)}
    if kind == "adjoint" and c["steps"] * c["n"] ** 3 <= 10 * 64 ** 3:
        n = c["n"]
        S = _clean(_adjoint_field(n, seed)).requires_grad_(True)
        X = S
        for dt in _adjoint_dts(c):
            X = checkpoint(_step, X, float(dt), 1.0 / n, {"ppm": 1}, BCS["periodic"], use_reentrant=False)
        loss = 0.5 * ((X[0] - _adjoint_field(n, seed + 1)[0]) ** 2).sum()
        return {"rho": X[0].detach(), "grad": [torch.autograd.grad(loss, S)[0]]}
    return None
