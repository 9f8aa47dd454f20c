"""The work that models built on this library have it do, as cases to time.

Five kinds of work, each through the entry points of ``orctm_amd.nh`` that a model calls:

* ``solve``: ``NHSolver.solve(DIVG, PNH)``, the drop-in for ``petsc_solve_3D`` of every time step, on the
  caller's Fortran arrays, from a zero guess;
* ``step``: the whole nonhydrostatic part of a time step: ``divergence`` from the velocities, the
  resident solve, ``project`` back onto the velocities;
* ``batch``: uneven independent systems (ensemble members, nests) advanced by one ``NHBatch.solve``;
* ``serve``: requests of several warm-started time steps each through ``NHServer``;
* ``surface``: ``NHBarotropic.troneu``, the barotropic free-surface solve of every time step.

Two recipes of basin. ``ocean``: a regional tile, dx = 1.85 km, 5 to 250 m layers over 5000 m, smoothed
random bathymetry with 25 % land and partial bottom cells, open boundaries (or periodic along x, closed
north and south, with ``cyclic``). ``tank``: the internal-solitary-wave transect, dx = 50 m, 2 to 40 m
layers over 1500 m, a Gaussian ridge, periodic along y, closed ends.
"""
import math

import numpy as np
import torch

from orctm_amd import abi, synth
from orctm_amd.nh import NHBarotropic, NHBatch, NHServer, NHSolver, options

PRECISION = {"mixed": abi.MIXED, "fp64": abi.FP64}

# PCG iterations a solve of a recipe takes to 1e-10, for work()
OCEAN_ITERATIONS = 42
TANK_ITERATIONS = 490  # at 512 columns along the transect, in proportion to them


def listed():
    return [
        # the 2-D ISW transect of the model's verification cases, in the reference's precision and in mixed:
        # few columns, many levels, many iterations; launches and latency are what counts
        {"name": "transect_fp64", "kind": "solve", "basin": "tank", "nx": 512, "ny": 4, "nz": 100, "precision": "fp64"},
        {"name": "transect_mixed", "kind": "solve", "basin": "tank", "nx": 512, "ny": 4, "nz": 100, "precision": "mixed"},
        # a small nest: the smallest grid that the serving workload sends
        {"name": "nest_small_mixed", "kind": "solve", "basin": "ocean", "nx": 128, "ny": 128, "nz": 30,
         "precision": "mixed"},
        # a ragged nest (odd sizes, nothing a multiple of a tile) in the reference's precision
        {"name": "nest_ragged_fp64", "kind": "solve", "basin": "ocean", "nx": 203, "ny": 194, "nz": 35,
         "precision": "fp64"},
        # an ordinary regional grid
        {"name": "regional_mid_mixed", "kind": "solve", "basin": "ocean", "nx": 512, "ny": 443, "nz": 49,
         "precision": "mixed"},
        # the regional tile of the headline benchmark
        {"name": "regional_mixed", "kind": "solve", "basin": "ocean", "nx": 1024, "ny": 768, "nz": 60,
         "precision": "mixed"},
        # a large ragged regional grid in the reference's precision
        {"name": "regional_fp64", "kind": "solve", "basin": "ocean", "nx": 813, "ny": 671, "nz": 58, "precision": "fp64"},
        # the nonhydrostatic part of a whole time step on a nest: right-hand side, solve, projection
        {"name": "step_mixed", "kind": "step", "basin": "ocean", "nx": 323, "ny": 293, "nz": 42, "precision": "mixed"},
        # an ensemble of nests of uneven sizes, advanced together
        {"name": "batch_mixed", "kind": "batch", "basin": "ocean", "members": 8, "lo": 96, "hi": 512, "nz_lo": 30,
         "nz_hi": 60, "precision": "mixed"},
        # a burst of requests on the serving loop, three sizes of grid, several warm-started steps each
        {"name": "serve_mixed", "kind": "serve", "basin": "ocean", "requests": 9, "steps": 4, "classes": 3,
         "precision": "mixed"},
        # the free surface of the regional tile, and that of the transect
        {"name": "surface_regional", "kind": "surface", "basin": "ocean", "nx": 1024, "ny": 768, "sweeps": 250},
        {"name": "surface_transect", "kind": "surface", "basin": "tank", "nx": 512, "ny": 4, "sweeps": 250},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    largest = _cost(next(c for c in listed() if c["name"] == "regional_mixed"))
    while True:
        kind = rng.choice(("solve", "solve", "solve", "tank", "step", "batch", "serve", "surface"))
        precision = rng.choice(("mixed", "fp64"))
        if kind == "tank":
            c = {"kind": "solve", "basin": "tank", "nx": _log_int(rng, 128, 1024), "ny": rng.choice((3, 4, 5, 8)),
                 "nz": rng.randint(40, 120), "precision": precision}
        elif kind in ("solve", "step"):
            c = {"kind": kind, "basin": "ocean", "nx": _log_int(rng, 96, 1024), "ny": _log_int(rng, 96, 768),
                 "nz": rng.randint(30, 60), "precision": precision, "cyclic": rng.random() < 0.2}
            if kind == "step" and c["nx"] * c["ny"] * c["nz"] > 12_000_000:
                continue
        elif kind == "batch":
            c = {"kind": "batch", "basin": "ocean", "members": rng.randint(2, 12), "lo": 96,
                 "hi": _log_int(rng, 128, 512), "nz_lo": 30, "nz_hi": 60, "precision": precision}
        elif kind == "serve":
            c = {"kind": "serve", "basin": "ocean", "requests": rng.randint(4, 16), "steps": rng.randint(2, 6),
                 "classes": rng.randint(1, 3), "precision": "mixed"}
        else:
            tank = rng.random() < 0.3
            c = {"kind": "surface", "basin": "tank" if tank else "ocean", "nx": _log_int(rng, 96, 1024),
                 "ny": rng.choice((3, 4, 5, 8)) if tank else _log_int(rng, 96, 768), "sweeps": 250}
        if _cost(c) <= largest:
            return c


# ---- inputs -----------------------------------------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _rng(seed, stream):
    g = torch.Generator(device=_device())
    g.manual_seed((int(seed) * 1_000_003 + stream) % (1 << 62))
    return g


def _normal(seed, stream, *shape):
    return torch.randn(*shape, generator=_rng(seed, stream), device=_device(), dtype=torch.float64)


def _spec(basin, nx, ny, nz, cyclic=False):
    if basin == "tank":
        return synth.GridSpec(nx, ny, nz, dx=50.0, dy=50.0, dz0=2.0, dz1=40.0, depth=1500.0, bathy="ridge",
                              ridge_height=800.0, ridge_width=5000.0, cyclic_y=True, open_w=False, open_e=False,
                              open_n=False, open_s=False, frac_lo=0.2, sigma_u=0.1)
    if cyclic:
        return synth.GridSpec(nx, ny, nz, cyclic_x=True, open_n=False, open_s=False)
    return synth.GridSpec(nx, ny, nz)


def _halo(a, spec, closed):
    """The halo ring of a (JE, IE) field: periodic, else open (the boundary column again), else `closed`."""
    if spec.cyclic_x:
        a[:, 0], a[:, -1] = a[:, -2].clone(), a[:, 1].clone()
    else:
        a[:, 0] = a[:, 1] if spec.open_w else closed
        a[:, -1] = a[:, -2] if spec.open_e else closed
    if spec.cyclic_y:
        a[0, :], a[-1, :] = a[-2, :].clone(), a[1, :].clone()
    else:
        a[0, :] = a[1, :] if spec.open_n else closed
        a[-1, :] = a[-2, :] if spec.open_s else closed


class _Sea:
    """One basin's arrays as tensors, k slowest and i fastest: the caller's Fortran arrays as they lie in memory."""

    def __init__(self, spec, seed):
        self.spec = spec
        nx, ny, nz = spec.nx, spec.ny, spec.nz
        self.IE, self.JE, self.KE = nx + 2, ny + 2, nz
        dev, f8 = _device(), torch.float64
        self.dzw = torch.tensor(synth.stretched_dzw(nz, spec.dz0, spec.dz1, spec.depth), dtype=f8, device=dev)
        self.tiestw = torch.cat([torch.zeros(1, dtype=f8, device=dev), torch.cumsum(self.dzw, 0)])
        self.tiestu = torch.cat([0.5 * (self.tiestw[:-1] + self.tiestw[1:]), torch.tensor([9000.0], dtype=f8, device=dev)])
        full = lambda nj, ni, v: torch.full((nj, ni), v, dtype=f8, device=dev)  # noqa: E731
        self.dlxp, self.dlyp = full(self.JE, self.IE, spec.dx), full(self.JE, self.IE, spec.dy)
        self.dlxu, self.dlyv = full(self.JE, self.IE + 1, spec.dx), full(self.JE + 1, self.IE, spec.dy)
        self.depto = full(self.JE, self.IE, 0.0)
        if spec.bathy == "ridge":
            x = (torch.arange(self.IE, dtype=f8, device=dev) - 0.5) * spec.dx
            self.depto[:] = spec.depth - spec.ridge_height * torch.exp(-(((x - 0.5 * nx * spec.dx) / spec.ridge_width) ** 2))
        else:
            ky, kx = torch.fft.fftfreq(ny, dtype=f8, device=dev), torch.fft.rfftfreq(nx, dtype=f8, device=dev)
            smooth = torch.exp(-2.0 * (math.pi * spec.smooth) ** 2 * (ky[:, None] ** 2 + kx[None, :] ** 2))
            field = torch.fft.irfft2(torch.fft.rfft2(_normal(seed, 11, ny, nx)) * smooth, s=(ny, nx))
            ranks = torch.empty(nx * ny, dtype=f8, device=dev)
            ranks[torch.argsort(field.reshape(-1), stable=True)] = torch.arange(nx * ny, dtype=f8, device=dev)
            land = spec.land_frac * nx * ny
            deep = spec.dmin + (spec.dmax - spec.dmin) * (ranks - land) / max(nx * ny - 1 - land, 1.0)
            self.depto[1:-1, 1:-1] = torch.where(ranks < land, torch.zeros_like(deep), deep).reshape(ny, nx)
        _halo(self.depto, spec, 0.0)
        part = full(self.JE, self.IE, 1.0)
        part[1:-1, 1:-1] = 1.0 - torch.rand(ny, nx, generator=_rng(seed, 23), device=dev, dtype=f8) * (1.0 - spec.frac_lo)
        _halo(part, spec, 1.0)
        bottom = torch.searchsorted(self.tiestu[:nz].contiguous(), self.depto)  # wet levels of each column
        level = torch.arange(nz, device=dev)[:, None, None]
        self.weto = (level < bottom).to(f8)
        self.ddpo = torch.where(level < bottom - 1, self.dzw[:, None, None], torch.zeros((), dtype=f8, device=dev))
        self.ddpo = torch.where(level == bottom - 1, part * self.dzw[:, None, None], self.ddpo)

    def grid(self):
        g = synth.Grid(self.spec, _host(self.dzw), *(_host(t) for t in (
            self.dlxp, self.dlyp, self.dlxu, self.dlyv, self.ddpo, self.weto)))
        return g

    def divg(self, seed):
        """DIVG of a random velocity field masked to the wet faces, with a time step of 1."""
        s, w = self.spec.sigma_u, self.weto
        u = torch.zeros(self.KE, self.JE, self.IE + 1, dtype=torch.float64, device=w.device)
        u[:, :, 1:-1] = s * _normal(seed, 31, self.KE, self.JE, self.IE - 1) * w[:, :, :-1] * w[:, :, 1:]
        out = (u[:, :, 1:] - u[:, :, :-1]) / self.dlxp
        u = torch.zeros(self.KE, self.JE + 1, self.IE, dtype=torch.float64, device=w.device)
        u[:, 1:-1] = s * _normal(seed, 37, self.KE, self.JE - 1, self.IE) * w[:, :-1] * w[:, 1:]
        out += (u[:, :-1] - u[:, 1:]) / self.dlyp
        u = torch.zeros(self.KE + 1, self.JE, self.IE, dtype=torch.float64, device=w.device)
        u[:-1] = s * _normal(seed, 41, self.KE, self.JE, self.IE) * w
        u[1:-1] *= w[:-1]
        out += (u[:-1] - u[1:]) / self.ddpo.clamp(min=1.0e-3)
        return out


def _host(t):
    """A tensor as the Fortran array with the same memory."""
    return t.cpu().numpy().T


def _faces(sea):
    """Depths at u- and v-points: the shallower of the two neighbours, end faces copied."""
    d, spec = sea.depto, sea.spec
    u = torch.zeros(sea.JE, sea.IE + 1, dtype=d.dtype, device=d.device)
    u[:, 1:-1] = torch.minimum(d[:, :-1], d[:, 1:])
    u[:, 0], u[:, -1] = u[:, 1], u[:, -2]
    _exchange(u[None], spec, 0, 1)
    v = torch.zeros(sea.JE + 1, sea.IE, dtype=d.dtype, device=d.device)
    v[1:-1] = torch.minimum(d[:-1], d[1:])
    v[0], v[-1] = v[1], v[-2]
    _exchange(v[None], spec, 1, 0)
    return u, v


def _exchange(a, spec, i0, j0):
    """Periodic copies of a (k, j0:JE, i0:IE) field, in place: x first, then y."""
    IE = spec.nx + 2
    if spec.cyclic_x:
        first, last = a[:, :, 2 - i0].clone(), a[:, :, IE - 1 - i0].clone()
        a[:, :, 1 - i0], a[:, :, IE - i0] = last, first
    if spec.cyclic_y:
        first, last = a[:, 1].clone(), a[:, -2].clone()
        a[:, 0], a[:, -1] = last, first


def _velocity(sea, seed, dt=60.0):
    """Velocity-side metrics and velocities of a step, as tensors by the names of the model's arrays."""
    spec, K, J, I = sea.spec, sea.KE, sea.JE, sea.IE  # noqa: E741
    v = {n: getattr(sea, n) for n in ("dlxp", "dlyp", "ddpo", "weto")}
    du, dv = _faces(sea)

    def layers(d):
        top, mid, below = sea.tiestw[:-1, None, None], sea.tiestu[:-1, None, None], sea.tiestu[1:, None, None]
        zero = torch.zeros((), dtype=d.dtype, device=d.device)
        return torch.where(below < d, sea.dzw[:, None, None], torch.where(mid < d, d - top, zero))

    v["dduo"], v["ddue"] = layers(du), layers(dv)
    v["amsuo"], v["amsue"] = (v["dduo"] > 0).to(du.dtype), (v["ddue"] > 0).to(du.dtype)
    v["dlyu"] = torch.full_like(sea.dlxu, spec.dy)
    v["dlxv"] = torch.full_like(sea.dlyv, spec.dx)
    v["dtdxpo"], v["dtdyo"], v["dtdxuo"], v["dpye"] = dt / sea.dlxp, dt / sea.dlyp, dt / sea.dlxu, dt / sea.dlyv
    s, wet_top = spec.sigma_u, torch.cat([sea.weto, torch.zeros_like(sea.weto[:1])])
    for name, stream in (("uoo", 61), ("uoo_1", 62)):
        v[name] = s * _normal(seed, stream, K, J, I + 1) * v["amsuo"]
        _exchange(v[name], spec, 0, 1)
    for name, stream in (("voe", 63), ("voe_1", 64)):
        v[name] = s * _normal(seed, stream, K, J + 1, I) * v["amsue"]
        _exchange(v[name], spec, 1, 0)
    for name, stream in (("wno", 65), ("wno_1", 66)):
        v[name] = 0.01 * s * _normal(seed, stream, K + 1, J, I) * wet_top
        _exchange(v[name], spec, 1, 1)
    v["zo"] = 0.5 * _normal(seed, 67, J, I) * sea.weto[0]
    _exchange(v["zo"][None], spec, 1, 1)
    return v


METRICS = ("dlxp", "dlyp", "ddpo", "weto", "amsuo", "dduo", "dtdxuo", "dlyu", "amsue", "ddue", "dpye", "dlxv", "dtdxpo",
           "dtdyo")
VELOCITY = ("uoo", "uoo_1", "voe", "voe_1", "wno", "wno_1", "zo")


def _surface(case, seed):
    """Metrics, constants and barotropic velocities of the free-surface solve, as tensors."""
    sea = _Sea(_spec(case["basin"], case["nx"], case["ny"], 60), seed)
    spec = sea.spec
    dt = 60.0 if case["basin"] == "ocean" else 10.0
    b = {"dlxp": sea.dlxp, "dlyp": sea.dlyp, "dtdxpo": dt / sea.dlxp, "dtdyo": dt / sea.dlyp, "weto1": sea.weto[0],
         "dlxu": sea.dlxu, "dlyu": torch.full_like(sea.dlxu, spec.dy), "dlxv": torch.full_like(sea.dlyv, spec.dx),
         "dlyv": sea.dlyv}
    b["deuto"], b["deute"] = _faces(sea)
    mu, mv = (b["deuto"] > sea.tiestu[0]).to(torch.float64), (b["deute"] > sea.tiestu[0]).to(torch.float64)
    for name, stream in (("u1o", 81), ("uzo", 82)):
        b[name] = spec.sigma_u * _normal(seed, stream, sea.JE, sea.IE + 1) * mu
        _exchange(b[name][None], spec, 0, 1)
    for name, stream in (("v1e", 83), ("vze", 84)):
        b[name] = spec.sigma_u * _normal(seed, stream, sea.JE + 1, sea.IE) * mv
        _exchange(b[name][None], spec, 1, 0)
    return sea, b, {"g": 9.81, "conn": 0.5, "cono": 0.5, "stabn": 0.6, "dt": dt, "sorpar": 1.75}


def _members(case, seed):
    """The systems of a batch: sizes spread over the case's ranges by the place in the batch, seeds of their own."""
    out = []
    for m in range(case["members"]):
        x, y, z = ((m * g + 0.35) % 1.0 for g in (0.6180339887, 0.7548776662, 0.5698402910))
        n = lambda t, lo, hi: lo + int(t * (hi - lo + 1))  # noqa: E731
        out.append((_spec(case["basin"], n(x, case["lo"], case["hi"]), n(y, case["lo"], case["hi"]),
                          n(z, case["nz_lo"], case["nz_hi"])), seed + 101 * m))
    return out


def _classes(case, seed):
    """The grids of the serving case: the smallest sizes of the serving workload's ladder."""
    return [(_spec(case["basin"], *synth.config5_size(m / 6.0)), seed + 101 * m) for m in range(case["classes"])]


AMPLITUDE = 0.01  # relative change of the right-hand side between a request's steps


# ---- a pass -----------------------------------------------------------------------------------------


def _solver(sea, precision):
    return NHSolver(sea.grid(), options(precision=PRECISION[precision], warm_start=False))


def _zeros(grid):
    return np.zeros((grid.IE, grid.JE, grid.KE), order="F")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "surface":
        sea, fields, constants = _surface(case, seed)
        b = synth.BarotropicState()
        b.IE, b.JE, b.i_start, b.j_start = sea.IE, sea.JE, 0, 0
        b.cyc_x, b.cyc_y, b.iterations = sea.spec.cyclic_x, sea.spec.cyclic_y, case["sweeps"]
        for name, t in fields.items():
            setattr(b, name, _host(t))
        for name, x in constants.items():
            setattr(b, name, x)
        flat = (sea.IE, sea.JE)
        return {"kind": kind, "solver": NHBarotropic(b), "b": b, "b1o": np.zeros(flat, order="F"),
                "z1o": np.zeros(flat, order="F")}
    if kind == "solve":
        sea = _Sea(_spec(case["basin"], case["nx"], case["ny"], case["nz"], case.get("cyclic", False)), seed)
        s = _solver(sea, case["precision"])
        return {"kind": kind, "solver": s, "divg": _host(sea.divg(seed)), "pnh": _zeros(s.grid)}
    if kind == "step":
        sea = _Sea(_spec(case["basin"], case["nx"], case["ny"], case["nz"], case.get("cyclic", False)), seed)
        s = _solver(sea, case["precision"])
        v, state = _velocity(sea, seed), synth.VelocityState()
        for name in METRICS + VELOCITY:
            setattr(state, name, _host(v[name]))
        state.dt, state.dti = 60.0, 1.0 / 60.0
        s.attach_vgrid(state)
        return {"kind": kind, "solver": s, "v": state, "pnh": _zeros(s.grid), "uoo": np.empty_like(state.uoo),
                "voe": np.empty_like(state.voe), "wno": np.zeros_like(state.wno)}
    systems = _members(case, seed) if kind == "batch" else _classes(case, seed)
    solvers = []
    for spec, own in systems:
        sea = _Sea(spec, own)
        solvers.append(_solver(sea, case["precision"]) if kind == "batch" else
                       NHSolver(sea.grid(), options(precision=PRECISION[case["precision"]])))
        if kind == "batch":
            solvers[-1].divg = _host(sea.divg(own))
        else:
            solvers[-1].set_rhs(_host(sea.divg(own)))
    if kind == "batch":
        return {"kind": kind, "solvers": solvers, "batch": NHBatch(solvers), "pnh": [_zeros(s.grid) for s in solvers]}
    owner = [solvers[r % len(solvers)] for r in range(case["requests"])]
    return {"kind": kind, "owner": owner, "steps": case["steps"], "seed": seed, "server": NHServer(),
            "pnh": [_zeros(s.grid) for s in owner]}


def run(state):
    kind = state["kind"]
    if kind == "surface":
        b = state["b"]
        state["solver"].troneu(b.u1o, b.uzo, b.v1e, b.vze, state["b1o"], state["z1o"])
        return {"z1o": state["z1o"], "b1o": state["b1o"]}
    if kind == "solve":
        state["solver"].solve(state["divg"], state["pnh"])
        return state["pnh"]
    if kind == "step":
        s, v = state["solver"], state["v"]
        s.divergence(v.uoo, v.uoo_1, v.voe, v.voe_1, v.wno, v.wno_1, v.zo)
        s.solve_resident()
        # the correction changes the velocities in place; the model keeps the uncorrected ones beside them
        np.copyto(state["uoo"], v.uoo)
        np.copyto(state["voe"], v.voe)
        s.project(state["pnh"], state["uoo"], state["voe"], state["wno"])
        return {n: state[n] for n in ("pnh", "uoo", "voe", "wno")}
    if kind == "batch":
        for s in state["solvers"]:
            s.set_rhs(s.divg)
        state["batch"].solve()
        for s, p in zip(state["solvers"], state["pnh"]):
            s.get_solution(p)
        return state["pnh"]
    server = state["server"]
    tickets = [server.submit(m, state["steps"], perturb=AMPLITUDE, seed=state["seed"] + 1000 * r, out=p)
               for r, (m, p) in enumerate(zip(state["owner"], state["pnh"]))]
    for t in tickets:
        server.wait(t)
    return state["pnh"]


# ---- what a pass cannot do without ------------------------------------------------------------------


def _sizes(case):
    """(cells, iterations) of each system solved in a pass of a case, one entry per solve."""
    if case["kind"] == "batch":
        return [(s.cells, OCEAN_ITERATIONS) for s, _ in _members(case, 0)]
    if case["kind"] == "serve":
        grids = [s.cells for s, _ in _classes(case, 0)]
        return [(grids[r % len(grids)], OCEAN_ITERATIONS) for r in range(case["requests"]) for _ in range(case["steps"])]
    its = OCEAN_ITERATIONS if case["basin"] == "ocean" else TANK_ITERATIONS * case["nx"] / 512.0
    return [(case["nx"] * case["ny"] * case["nz"], its)]


def _cost(case):
    return work(case)["bytes"]


def work(case):
    """Bytes: the host arrays in and out once, and per iteration the solution, the residual and the search
    direction read and written once in the working precision (a surface solve: its iterate once a sweep)."""
    if case["kind"] == "surface":
        n = (case["nx"] + 2) * (case["ny"] + 2)
        return {"bytes": 8.0 * n * 7 + 16.0 * n * case["sweeps"], "flops": 11.0 * n * case["sweeps"]}
    word = 4 if case["precision"] == "mixed" else 8
    cells = sum(n for n, _ in _sizes(case))
    cell_its = sum(n * its for n, its in _sizes(case))
    host = {"solve": 16, "step": 8 * 12, "batch": 16, "serve": 16}[case["kind"]]
    return {"bytes": float(host * cells + 6 * word * cell_its), "flops": 30.0 * cell_its}


# ---- the values in 64 bits, by plain torch ------------------------------------------------------------


class _Operator:
    """The 7-point pressure operator of a basin in 64 bits, and PCG on S(-A) with a solve of each column as
    the preconditioner, S = DLXP*DLYP/ZP, restarted on the true residual until it stops falling."""

    def __init__(self, sea):
        spec, K = sea.spec, sea.KE
        d, w, dz = sea.ddpo, sea.weto, sea.dzw
        inner = (slice(None), slice(1, -1), slice(1, -1))
        d, here = d[inner], w[inner]
        mid = torch.where(d[:-1] == 0, ((dz[1:] + dz[:-1]) / 2)[:, None, None],
                          torch.where(d[1:] == 0, d[:-1], (d[:-1] + d[1:]) / 2))
        top = torch.where(d[:1] == 0, dz[0] / 2, d[:1] / 2)
        low = torch.where(d[-1:] == 0, dz[-1], d[-1:])
        zw = 1 / torch.cat([top, mid, low])
        zp = 2 / (1 / zw[:-1] + 1 / zw[1:])
        p = (slice(1, -1), slice(1, -1))
        xw, xe = 1 / (sea.dlxu[1:-1, 1:-2] * sea.dlxp[p]), 1 / (sea.dlxu[1:-1, 2:-1] * sea.dlxp[p])
        yn, ys = 1 / (sea.dlyv[1:-2, 1:-1] * sea.dlyp[p]), 1 / (sea.dlyv[2:-1, 1:-1] * sea.dlyp[p])
        ww, we, wn, ws = w[:, 1:-1, :-2], w[:, 1:-1, 2:], w[:, :-2, 1:-1], w[:, 2:, 1:-1]
        west, east, north, south = here * ww * xw, here * we * xe, here * wn * yn, here * ws * ys
        up, down = here * zw[:-1] * zp, torch.zeros_like(zp)
        below = torch.cat([here[1:], torch.zeros_like(here[:1])])
        down[:-1] = (here * below * zw[1:] * zp)[:-1]
        centre = ww * xw + we * xe + wn * yn + ws * ys + zw[:-1] * zp  # no flux through land or the bottom ...
        centre += torch.where(below != 0, zw[1:] * zp, torch.zeros_like(zp))
        if K > 0:  # ... but the surface row takes both its faces whatever lies below
            centre[0] = (ww * xw + we * xe + wn * yn + ws * ys)[0] + (zw[0] + zw[1]) * zp[0]
        dry = (xw + xe + yn + ys) + (zw[:-1] + zw[1:]) * zp
        centre = torch.where(here != 0, centre, dry)
        up[0] = 0
        if not spec.cyclic_x:
            west[:, :, 0] = 0
            east[:, :, -1] = 0
        if not spec.cyclic_y:
            north[:, 0] = 0
            south[:, -1] = 0
        self.wet, self.c = here, (-centre, west, east, north, south, up, down)
        scale = sea.dlxp[p] * sea.dlyp[p] / zp
        self.scale, e = scale, -scale * up
        self.l, self.inv = [None] * K, [None] * K
        for k in range(K):
            diag = scale[k] * centre[k]
            if k:
                link = torch.where(down[k - 1] != 0, e[k], torch.zeros_like(e[k]))
                self.l[k] = link * self.inv[k - 1]
                diag = diag - self.l[k] * link
            self.inv[k] = 1 / diag

    def times(self, x):
        c, w, e, n, s, u, d = self.c
        y = c * x
        y += w * torch.roll(x, 1, 2)
        y += e * torch.roll(x, -1, 2)
        y += n * torch.roll(x, 1, 1)
        y += s * torch.roll(x, -1, 1)
        y[1:] += u[1:] * x[:-1]
        y[:-1] += d[:-1] * x[1:]
        return y

    def column_solve(self, r):
        z = torch.empty_like(r)
        z[0] = r[0]
        for k in range(1, len(self.l)):
            torch.addcmul(r[k], self.l[k], z[k - 1], value=-1, out=z[k])
        z[-1] *= self.inv[-1]
        for k in range(len(self.l) - 2, -1, -1):
            z[k] *= self.inv[k]
            z[k].addcmul_(self.l[k + 1], z[k + 1], value=-1)
        return z

    def solve(self, b):
        b = b * self.wet
        x, best = torch.zeros_like(b), None
        size = float(b.norm())
        if size == 0:
            return x
        for _ in range(6):
            t = b - self.times(x)
            rel = float(t.norm()) / size
            if best is not None and rel > 0.5 * best[0]:
                break
            best = (rel, x.clone())
            if rel < 1e-15:
                break
            r, y, p, rz = -self.scale * t, torch.zeros_like(b), None, None
            goal, it = 1e-6 * float(r.norm()), 0
            while it < 6000:
                z = self.column_solve(r)
                new = torch.sum(r * z)
                p = z if p is None else z + (new / rz) * p
                rz = new
                q = self.times(p)
                q *= -self.scale
                a = rz / torch.sum(p * q)
                y += a * p
                r -= a * q
                it += 1
                if it % 4 == 0 and float(r.norm()) <= goal:
                    break
            x = x + y
        return best[1]


def _whole(sea, x):
    """An interior solution in the caller's array, its halo 0."""
    out = torch.zeros(sea.KE, sea.JE, sea.IE, dtype=x.dtype, device=x.device)
    out[:, 1:-1, 1:-1] = x
    return out


def _perturbation(cells, seed):
    """N(0, 1) per cell from the counter-based stream of orctm_nh_perturb_rhs."""
    def wrap(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    def shift(z, n):
        return (z >> n) & ((1 << (64 - n)) - 1)

    def mix(z):
        z = z + wrap(0x9E3779B97F4A7C15)
        z = (z ^ shift(z, 30)) * wrap(0xBF58476D1CE4E5B9)
        z = (z ^ shift(z, 27)) * wrap(0x94D049BB133111EB)
        return z ^ shift(z, 31)

    key = mix(torch.tensor(wrap(seed), dtype=torch.int64, device=_device()))
    n = torch.arange(cells, dtype=torch.int64, device=_device())
    u1 = 1.0 - shift(mix(key + 2 * n), 11).double() * (1.0 / 9007199254740992.0)
    u2 = shift(mix(key + 2 * n + 1), 11).double() * (1.0 / 9007199254740992.0)
    return torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)


def _exact_step(sea, seed):
    v, dt, spec = _velocity(sea, seed), 60.0, sea.spec
    gu, gv, gw = ((v[n] - v[n + "_1"]) / dt for n in ("uoo", "voe", "wno"))
    h = sea.ddpo.clamp(min=1.0e-3)
    h[0] += v["zo"]
    divg = (gu[:, :, 1:] - gu[:, :, :-1]) / sea.dlxp + (gv[:, :-1] - gv[:, 1:]) / sea.dlyp + (gw[:-1] - gw[1:]) / h
    p = _whole(sea, _Operator(sea).solve(divg[:, 1:-1, 1:-1]))
    _exchange(p, spec, 1, 1)
    if not spec.cyclic_x:
        if spec.open_w:
            p[:, 1:-1, 0] = p[:, 1:-1, 1]
        if spec.open_e:
            p[:, 1:-1, -1] = p[:, 1:-1, -2]
    if not spec.cyclic_y:
        if spec.open_n:
            p[:, 0] = p[:, 1]
        if spec.open_s:
            p[:, -1] = p[:, -2]
    u, w = v["uoo"].clone(), v["voe"].clone()
    face = (slice(None), slice(1, -1), slice(1, -1))
    u[face] += v["amsuo"][face] * v["dtdxuo"][1:-1, 1:-1] * (p[:, 1:-1, :-1] - p[:, 1:-1, 1:])
    w[face] += v["amsue"][face] * v["dpye"][1:-1, 1:-1] * (p[:, 1:, 1:-1] - p[:, :-1, 1:-1])
    _exchange(u, spec, 0, 1)
    _exchange(w, spec, 1, 0)
    fu, fv = u * v["dduo"] * v["dlyu"], w * v["ddue"] * v["dlxv"]
    gain = sea.weto / dt * (v["dtdxpo"] * (fu[:, :, :-1] - fu[:, :, 1:]) / sea.dlyp
                            + v["dtdyo"] * (fv[:, 1:] - fv[:, :-1]) / sea.dlxp)
    wno = torch.zeros(sea.KE + 1, sea.JE, sea.IE, dtype=u.dtype, device=u.device)
    wno[:-1] = torch.flip(torch.cumsum(torch.flip(gain, (0,)), 0), (0,))
    _exchange(wno, spec, 1, 1)
    return {"pnh": _host(p), "uoo": _host(u), "voe": _host(w), "wno": _host(wno)}


def _exact_surface(case, seed):
    sea, b, c = _surface(case, seed)
    spec, half = sea.spec, c["g"] * c["conn"] * c["stabn"] * c["dt"] ** 2
    area = sea.dlxp * sea.dlyp
    uf, vf = b["deuto"] * b["dlyu"] / b["dlxu"] * half, b["deute"] * b["dlxv"] / b["dlyv"] * half
    ff = 1 / (area + uf[:, 1:] + uf[:, :-1] + vf[1:] + vf[:-1])
    _exchange(ff[None], spec, 1, 1)
    tu = (c["cono"] * b["u1o"] + c["conn"] * b["uzo"]) * b["dlyu"]
    tv = (c["cono"] * b["v1e"] + c["conn"] * b["vze"]) * b["dlxv"]
    b1o = b["weto1"] * (b["dtdxpo"] * (tu[:, :-1] - tu[:, 1:]) / sea.dlyp
                        + b["dtdyo"] * (tv[1:] - tv[:-1]) / sea.dlxp) * area
    z = torch.zeros_like(b1o)
    for edge in ((slice(None), 0), (slice(None), -1), (0, slice(None)), (-1, slice(None))):
        z[edge] = b1o[edge] / area[edge]
    j = torch.arange(2, sea.JE, device=z.device)[:, None]
    i = torch.arange(2, sea.IE, device=z.device)[None, :]
    inner = (slice(1, -1), slice(1, -1))
    for _ in range(case["sweeps"]):
        for colour in (0, 1):
            s = (b1o[inner] + uf[1:-1, 2:-1] * z[1:-1, 2:] + uf[1:-1, 1:-2] * z[1:-1, :-2]
                 + vf[2:-1, 1:-1] * z[2:, 1:-1] + vf[1:-2, 1:-1] * z[:-2, 1:-1])
            new = c["sorpar"] * ff[inner] * s + (1 - c["sorpar"]) * z[inner]
            z[inner] = torch.where((i + j + colour) % 2 == 0, new, z[inner])
            _exchange(z[None], spec, 1, 1)
    return {"z1o": _host(z), "b1o": _host(b1o)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "surface":
        return _exact_surface(case, seed)
    if kind in ("solve", "step"):
        sea = _Sea(_spec(case["basin"], case["nx"], case["ny"], case["nz"], case.get("cyclic", False)), seed)
        if kind == "step":
            return _exact_step(sea, seed)
        return _host(_whole(sea, _Operator(sea).solve(sea.divg(seed)[:, 1:-1, 1:-1])))
    if kind == "batch":
        seas = [(_Sea(spec, own), own) for spec, own in _members(case, seed)]
        return [_host(_whole(s, _Operator(s).solve(s.divg(own)[:, 1:-1, 1:-1]))) for s, own in seas]
    seas = [(_Sea(spec, own), own) for spec, own in _classes(case, seed)]
    models = [(s, _Operator(s), s.divg(own)[:, 1:-1, 1:-1]) for s, own in seas]
    out = []
    for r in range(case["requests"]):
        s, a, b = models[r % len(models)]
        b = b * a.wet
        for step in range(1, case["steps"]):
            b = b * (1.0 + AMPLITUDE * _perturbation(b.numel(), seed + 1000 * r + step).reshape(b.shape))
        out.append(_host(_whole(s, a.solve(b))))
    return out
