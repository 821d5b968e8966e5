"""The calls whose speed counts, as a program of this framework makes them.

A pass advances resident flow fields by the steps between two outputs and
hands the fields back to the program (Solver.step, Solver.download), or takes
a batch of requests through the continuous-batching server (Server.submit to
Server.result).  The fields handed back are the cells of the domain (lower
bound 1), U, V, W, the pressure and every scalar; the precision form's fields
are 32-bit numbers and are kept as such.

Kinds of case
  flat      uniform grid, rough floor, free-slip top, passive scalars
  urban     512x512x128 with the 64-building array of the benchmark
  scenario  buildings of one dispersion request (mixed-radix grids)
  channel   turbulent channel on the stretched grid, spectral or multigrid
  abl       moist, buoyant boundary layer over a floor of given temperature
  requests  a queue of scenarios through the server

exact() restates the step in plain torch, 64 bits, for every kind but abl.
Solid bodies enter it as they enter a solver: by the masks and point lists
that a program hands to it (elmm_lists).
"""
import math
import os
import sys
import time

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-elmm_amd"))

from elmm_amd import capi, cases, serving, workloads  # noqa: E402

XY = [16, 18, 24, 27, 32, 36, 48, 54, 64, 72, 81, 96, 108, 128, 144, 162, 192, 256]  # 2^a 3^b
BITS = {"fp64": capi.FP64, "fp32r": capi.FP32_REFINED}


def listed():
    return [
        # the smallest calls: a test-size box stepped one output interval at
        # a time, diagnostics read after every step (launch and sync latency)
        dict(name="flat32_fp64_diag", kind="flat", nx=32, ny=32, nz=32, precision="fp64", steps=4, diag=True),
        # the reference's uniform 64^3 configuration, one second of flow
        dict(name="flat64_fp32r", kind="flat", nx=64, ny=64, nz=64, precision="fp32r", steps=20),
        dict(name="flat64_fp64", kind="flat", nx=64, ny=64, nz=64, precision="fp64", steps=20),
        # extents off every tile and off the powers of two, two scalars, the
        # time step from the CFL number (one synchronisation a step)
        dict(name="flat_ragged_vardt_fp64", kind="flat", nx=162, ny=54, nz=41, precision="fp64", steps=10,
             nscalars=2, variable_dt=True),
        # one dispersion scenario, the size a serving queue sees most
        dict(name="scenario_1m4_fp32r", kind="scenario", cells=1400000, precision="fp32r", steps=40),
        # the turbulent channel, stretched z: spectral and multigrid pressure
        dict(name="channel256_fp32r", kind="channel", nx=256, ny=128, nz=128, precision="fp32r", steps=40),
        dict(name="channel128_mg_fp64", kind="channel", nx=128, ny=64, nz=64, precision="fp64", steps=4,
             multigrid=True),
        # every physics option at once: temperature, moisture, wall laws
        dict(name="abl128_fp64", kind="abl", nx=128, ny=128, nz=64, precision="fp64", steps=10),
        # requests of several sizes at once: upload, projection, steps, result
        dict(name="requests6_fp32r", kind="requests", n=6, cells_min=250000, cells_max=1500000, precision="fp32r",
             steps=20),
        # the benchmark: street canyons at 33.5 M cells, both forms
        dict(name="urban512_fp32r", kind="urban", nx=512, ny=512, nz=128, precision="fp32r", steps=60),
        dict(name="urban512_fp64", kind="urban", nx=512, ny=512, nz=128, precision="fp64", steps=30),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["flat", "flat", "flat", "scenario", "channel", "channel", "abl", "requests"])
    c = dict(kind=kind, precision="fp64" if kind == "abl" else rng.choice(["fp64", "fp32r"]),
             steps=int(round(_log(rng, 4, 40))))
    if kind == "scenario":
        return dict(c, cells=int(_log(rng, 1.5e5, 3e6)))
    if kind == "requests":
        lo = _log(rng, 5e4, 4e5)
        return dict(c, n=rng.randint(2, 8), cells_min=int(lo), cells_max=int(lo * rng.uniform(1, 4)))
    near = lambda v: min(XY, key=lambda x: abs(math.log(x / v)))  # noqa: E731
    c.update(nx=near(_log(rng, 16, 256)), ny=near(_log(rng, 16, 256)), nz=int(round(_log(rng, 9, 140))))
    if kind == "flat":
        c.update(nscalars=rng.randint(0, 2), variable_dt=rng.random() < 0.25, diag=rng.random() < 0.25)
    if kind == "channel" and c["nx"] % 2 == 0 and c["ny"] % 2 == 0 and rng.random() < 0.3:
        c.update(multigrid=True, steps=min(c["steps"], 6))
    return c


# ------------------------------------------------------------------ inputs
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _noise(g, shape, amp):
    """Uniform in -amp..amp, 32-bit values (what the restart files hold)."""
    return ((torch.rand(shape, generator=g, device=_device()) * 2 - 1) * amp).double()


def _host(t):
    """A (nz, ny, nx) tensor as the Fortran-ordered array the library takes."""
    return t.cpu().numpy().T


def _config(case):
    k, n = case["kind"], {a: case[a] for a in ("nx", "ny", "nz")}
    if k == "channel":
        cfg = cases.channel_config(**n, dt=2e-4 * min(1.0, 128.0 / n["nz"]), autotune=1,
                                   poisson_solver=capi.POISSON_MG if case.get("multigrid") else capi.POISSON_FFT)
    elif k == "abl":
        bc = [capi.PERIODIC] * 4
        cfg = cases.uniform_config(
            **n, dx=2.0, dt=0.1, nscalars=1, autotune=1, enable_buoyancy=1, grav_acc=9.81, temperature_ref=295.0,
            temp_btype=bc + [capi.DIRICHLET, capi.DIRICHLET], side_temp=[0, 0, 0, 0, 295.0, 299.0],
            enable_moisture=1, moisture_ref=0.01, moist_btype=bc + [capi.DIRICHLET, capi.NEUMANN],
            side_moist=[0, 0, 0, 0, 0.012, 0.0])
    else:
        opt = dict(variable_dt=1, cfl_target=0.4, dt_max=0.1, dt_min=1e-4) if case.get("variable_dt") else {}
        cfg = cases.uniform_config(**n, dx=1.0, dt=0.05, nscalars=case.get("nscalars", 1), autotune=1, **opt)
    return capi.with_precision(cfg, BITS[case["precision"]])


def _wind(case):
    return {"flat": (1.0, 0.1), "urban": (3.0, 0.3), "abl": (4.0, 0.4)}[case["kind"]]


def _fields(case, seed):
    """U, V, W and the active scalars as (nz+6, ny+6, nx+6) tensors."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    g = torch.Generator(device=_device())
    g.manual_seed(seed)

    def box(values):
        f = torch.zeros((nz + 6, ny + 6, nx + 6), dtype=torch.float64, device=_device())
        f[3:3 + values.shape[0], 3:3 + ny, 3:3 + nx] = values
        return f

    if case["kind"] == "channel":
        zw = torch.tensor(cases.channel_zw(nz), device=_device())
        zp, ze = (zw[1:] + zw[:-1]) / 2, zw[1:-1]

        def law(z):
            dp = torch.minimum(z, zw[-1] - z) / 1e-3
            return torch.where(dp < 11.0, dp, torch.log(dp) / 0.41 + 5.5)[:, None, None]

        return [box(law(zp) * (1 + _noise(g, (nz, ny, nx), 0.05))), box(law(zp) * _noise(g, (nz, ny, nx), 0.05)),
                box(law(ze) * _noise(g, (nz - 1, ny, nx), 0.05))], []
    u0, amp = _wind(case)
    vel = [box(u0 + _noise(g, (nz, ny, nx), amp)), box(_noise(g, (nz, ny, nx), amp)),
           box(_noise(g, (nz - 1, ny, nx), amp))]
    if case["kind"] != "abl":
        return vel, []
    prof = torch.linspace(293.0, 299.0, nz, dtype=torch.float64, device=_device())[:, None, None]
    return vel, [box(prof + _noise(g, (nz, ny, nx), 0.2)), box(0.01 + _noise(g, (nz, ny, nx), 0.001))]


def _source(case, seed, s=0):
    """Street-level point source of scalar s: the middle of a cell."""
    return (0.5 + (5 + 7 * seed + 3 * s) % case["nx"], 0.5 + (3 + 11 * seed + s) % case["ny"], 0.5, 1.0, s)


def _request_cells(case):
    """Cell counts of a queue's requests, from cells_min to cells_max."""
    lo, hi = math.log(case["cells_min"]), math.log(case["cells_max"])
    return [math.exp(lo + (hi - lo) * q / (case["n"] - 1)) for q in range(case["n"])]


def _bodies(case, seed):
    """Solid bodies and point sources of a case's grid."""
    if case["kind"] == "urban":
        return workloads.urban_obstacles(seed=seed), [(12.5, 12.5, 0.5, 1.0, 0)]
    if case["kind"] == "abl":
        return [], [(12.5, 12.5, 0.5, 1.0, 0)]
    return [], [_source(case, seed, s) for s in range(0 if case["kind"] == "channel" else case.get("nscalars", 1))]


class _State:
    pass


def prepare(case, seed):
    """What a program holds before the call: the case's masks and lists and a
    solver whose initial fields are projected (for a queue of requests: the
    scenarios, their fields on the host, and the server)."""
    st = _State()
    st.case, st.keep32 = case, case["precision"] == "fp32r"
    if case["kind"] == "requests":
        st.requests = [serving._prepare(1000 * seed + q, c, BITS[case["precision"]])
                       for q, c in enumerate(_request_cells(case))]
        st.server = capi.Server(100e9, max_active=case["n"], chunk_steps=10)
        return st
    if case["kind"] == "scenario":
        cfg, st.lists, fields = serving._prepare(seed, case["cells"], BITS[case["precision"]])
    else:
        cfg = _config(case)
        cub, src = _bodies(case, seed)
        st.lists = capi.Case(cfg, cuboids=cub, sources=src, device=True)
        vel, active = _fields(case, seed)
        zero = np.zeros(capi.ghosted_shape(cfg), order="F")
        fields = [_host(f) for f in vel] + [zero, [zero] * cfg.nscalars]
    st.cfg = cfg
    st.solver = capi.Solver(cfg, st.lists)
    cases.upload_initial(st.solver, cfg, fields)
    st.ids = {"U": capi.F_U, "V": capi.F_V, "W": capi.F_W, "Pr": capi.F_PR}
    st.ids.update({f"S{s}": capi.F_SCALAR + s for s in range(cfg.nscalars)})
    if case["kind"] == "abl":
        st.ids.update(T=capi.F_TEMPERATURE, Q=capi.F_MOISTURE)
        st.solver.upload(capi.F_TEMPERATURE, _host(active[0]))
        st.solver.upload(capi.F_MOISTURE, _host(active[1]))
    st.solver.init()
    return st


def run(st):
    case = st.case
    if case["kind"] == "requests":
        ids = [st.server.submit(cfg, lists, f, case["steps"]) for cfg, lists, f in st.requests]
        while any(st.server.progress()):
            time.sleep(0.0001)
        out = {}
        for q, i in enumerate(ids):
            u, v, w, p, s = st.server.result(i)
            for name, a in zip("UVWPS", (u, v, w, p, s[0])):
                out[f"{q}{name}"] = _keep(st, a[3:-3, 3:-3, 3:-3])
            st.server.release(i)
        return out
    s, cfg, out = st.solver, st.cfg, {}
    if case.get("diag"):
        for _ in range(case["steps"]):
            d = s.step(1)
        out.update(cfl=d.cfl, dt=d.dt, time=d.time)
    else:
        s.step(case["steps"], diag=False)
    for name, field in st.ids.items():
        out[name] = _keep(st, s.download(field, lb=1, shape=(cfg.nx, cfg.ny, cfg.nz)))
    return out


def _keep(st, a):
    return torch.from_numpy(a).to(torch.float32) if st.keep32 else a


def work(case):
    """Bytes: per stage the velocity, the pressure and the scalars read and
    written once (each stage ends in a pressure solve over the whole domain,
    so no state stays on chip), the solve's right-hand side and solution in
    64 bits, and the fields handed back.  Operations: counted from the
    scheme's formulas, about 400 a cell and stage, plus the transforms."""
    if case["kind"] in ("scenario", "requests"):
        n = 1 if case["kind"] == "scenario" else case["n"]
        cells = case["cells"] if n == 1 and "cells" in case else n * math.sqrt(case["cells_min"] * case["cells_max"])
        nsc = 1
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
        nsc = {"channel": 0, "abl": 3}.get(case["kind"], case.get("nscalars", 1))
    b = 4 if case["precision"] == "fp32r" else 8
    stages = 3 * case["steps"]
    return {"bytes": cells * (stages * (2 * b * (4 + nsc) + 16) + 8 * (4 + nsc)),
            "flops": cells * stages * (400 + 60 * nsc + 5 * math.log2(max(cells, 2)))}


# ------------------------------------------------------------ exact values
class _Points:
    """Index arithmetic on (nz+6, ny+6, nx+6) fields for the point lists of a
    case: (n, 3) arrays of 1-based i, j, k."""

    def __init__(self, cfg, lists):
        self.ext = (cfg.nx, cfg.ny, cfg.nz)
        self.off = (1, cfg.nx + 6, (cfg.nx + 6) * (cfg.ny + 6))
        masks = [torch.from_numpy(np.ascontiguousarray(m.T)).to(_device()) for m in lists.masks()]
        self.solid, self.types = masks[0] > 0, masks[1:]
        n = int(np.prod(lists.shape()))
        view = lists.view
        flat = lambda p, k, t: torch.from_numpy(capi._np(p, k, t)).to(_device())  # noqa: E731
        self.open = [(flat(view.scfl_mask[d], n, np.uint8) != 0).reshape(self.solid.shape) for d in range(3)]
        self.faces = [self.lin(flat(view.scfl_ijk[d], 3 * view.scfl_n[d], np.int32)) for d in range(3)]
        self.wall = []
        for q in range(18):
            if view.wm_n[q]:
                ijk, dist, z0 = lists.wm_list(q)
                p = torch.from_numpy(ijk).to(_device())
                self.wall.append((q, self.lin(p), torch.from_numpy(dist).to(_device()),
                                  torch.from_numpy(z0).to(_device())))
        self.floor = self.lin(torch.from_numpy(lists.wmp_list()[0]).to(_device()))
        self.taps = []
        for c in range(4):
            ijk, ptr, src, coef = lists.ib_list(c)
            t, s = (self.lin(torch.from_numpy(a).to(_device())) for a in (ijk, src))
            seg = torch.repeat_interleave(torch.arange(len(ijk)), torch.from_numpy(np.diff(ptr)).long()).to(_device())
            self.taps.append((t, s, seg, torch.from_numpy(coef).to(_device())))
        self.levels = self.rounds(*self.taps[3][:3])
        self.null = [self.lin(torch.from_numpy(lists.null_list(c)).to(_device())) for c in range(3)]
        self.src = (self.lin(flat(view.src_ijk, 3 * view.src_n, np.int32)),
                    flat(view.src_scalar, view.src_n, np.int32), flat(view.src_flux, view.src_n, np.float64))

    def lin(self, ijk):
        p = ijk.reshape(-1, 3).long() + 2
        return p[:, 0] + p[:, 1] * self.off[1] + p[:, 2] * self.off[2]

    def inside(self, p):
        """Whether the cells p are cells of the domain."""
        i, j, k = p % self.off[1] - 2, p // self.off[1] % (self.ext[1] + 6) - 2, p // self.off[2] - 2
        return (i >= 1) & (i <= self.ext[0]) & (j >= 1) & (j <= self.ext[1]) & (k >= 1) & (k <= self.ext[2])

    def add(self, f, p, v):
        ok = self.inside(p)
        f.view(-1).index_add_(0, p[ok], v[ok])

    def rounds(self, tgt, src, seg):
        """The round of each point of a loop whose points may read what
        earlier ones wrote: points of one round are independent."""
        t, s, g = tgt.tolist(), src.tolist(), seg.tolist()
        at, wrote, read, lev = 0, {}, {}, []
        for p, cell in enumerate(t):
            b = at
            while at < len(g) and g[at] == p:
                at += 1
            mine = s[b:at]
            v = max([wrote.get(q, 0) for q in mine] + [read.get(cell, 0), wrote.get(cell, 0)])
            lev.append(v)
            wrote[cell] = v + 1
            for q in mine:
                read[q] = max(read.get(q, 0), v + 1)
        return torch.tensor(lev, device=_device())

    def interpolate(self, c, f):
        t, s, seg, coef = self.taps[c]
        return torch.zeros(len(t), dtype=f.dtype, device=f.device).index_add_(0, seg, coef * f.view(-1)[s])

    def bodies(self, vel):
        """Velocities at the points next to bodies from their neighbours."""
        for c, f in enumerate(vel):
            f.view(-1)[self.taps[c][0]] = self.interpolate(c, f)

    def viscosity(self, f):
        t, s, seg, coef = self.taps[3]
        for v in range(int(self.levels.max()) + 1 if len(t) else 0):
            on = self.levels == v
            f.view(-1)[t[on]] = self.interpolate(3, f)[on]

    def mass(self, vel, h):
        """Mass sources of the faces next to bodies, folded into the domain."""
        q = torch.zeros_like(vel[0])
        nx, ny, nz = self.ext
        for c, f in enumerate(vel):
            t = self.taps[c][0]
            v = f.view(-1)[t] / h[c]
            q.view(-1).index_add_(0, t, v)
            q.view(-1).index_add_(0, t + self.off[c], -v)
        q[:, :, nx + 2] += q[:, :, 2]
        q[:, :, 3] += q[:, :, nx + 3]
        q[:, ny + 2] += q[:, 2]
        q[:, 3] += q[:, ny + 3]
        q[3] += q[2]
        q[nz + 2] += q[nz + 3]
        return q


class _Flow:
    """The step in 64 bits on (nz+6, ny+6, nx+6) tensors, interior 3..n+2:
    fourth-order (uniform z) or second-order (stretched z) advection,
    Smagorinsky viscosity, wall stresses, limited scalar advection, immersed
    bodies, three-stage Runge-Kutta with a projection in every stage."""

    RHO, BETA, ALPHA = (0.0, -17 / 60, -5 / 12), (8 / 15, 5 / 12, 3 / 4), (4 / 15, 1 / 15, 1 / 6)

    def __init__(self, cfg, vel, lists):
        self.c, self.n = cfg, (cfg.nz, cfg.ny, cfg.nx)
        nz = cfg.nz
        self.dx, self.dy, self.vz = cfg.dx, cfg.dy, bool(cfg.stretched_z)
        zw = {}
        for k in range(-3, nz + 4):
            if not self.vz:
                zw[k] = k * cfg.dz
            elif 0 <= k <= nz:
                zw[k] = cfg.zw[k]
        if self.vz:
            for k in (-1, -2, -3):
                zw[k] = 2 * zw[0] - zw[-k]
            for k in range(nz + 1, nz + 4):
                zw[k] = 2 * zw[nz - 1] - zw[2 * nz - 2 - k]
        zp = {k: (zw[k - 1] + zw[k]) / 2 for k in range(-2, nz + 4)}

        def col(f, lo=1, hi=nz):
            return torch.tensor([f(k) for k in range(lo, hi + 1)], dtype=torch.float64, device=_device())[:, None, None]

        self.zw, self.zp = zw, zp
        self.dzp, self.dzw = col(lambda k: zw[k] - zw[k - 1]), col(lambda k: zp[k + 1] - zp[k])
        self.dzf = col(lambda k: zp[k + 1] - zp[k], 0, nz)       # faces 0..nz
        self.dzu = col(lambda k: zw[k + 1] - zw[k], 0, nz)
        self.dz2 = col(lambda k: zp[k + 1] - zp[k - 1])
        self.dzw2 = col(lambda k: zw[k + 1] - zw[k - 1])
        self.pts = _Points(cfg, lists)
        self.U = [f.clone() for f in vel]
        zero = torch.zeros_like(vel[0])
        self.P, self.visc, self.tdiff = zero.clone(), zero.clone(), zero.clone()
        self.S = [zero.clone() for _ in range(cfg.nscalars)]
        self.N, self.NS = [0.0] * 3, [0.0] * cfg.nscalars
        self.ustar, self.time = {}, 0.0
        # projection of the start, viscosity (with the ghost values from
        # before it) and the frozen scalar diffusivity
        self.bound_velocity(self.U)
        self.project(self.U, 1.0, None)
        self.subgrid()
        self.tdiff = (self.visc - cfg.nu) / float(np.float32(0.6)) + cfg.nu_scalar
        for f in self.S:
            self.bound_scalar(f)
        self.walls()
        self.bound_velocity(self.U)
        self.pts.bodies(self.U)

    def at(self, f, di=0, dj=0, dk=0):
        nz, ny, nx = self.n
        return f[3 + dk:3 + dk + nz, 3 + dj:3 + dj + ny, 3 + di:3 + di + nx]

    def wrap(self, f):
        nz, ny, nx = self.n
        f[:, :, :3] = f[:, :, nx:nx + 3].clone()
        f[:, :, nx + 3:] = f[:, :, 3:6].clone()
        f[:, :3] = f[:, ny:ny + 3].clone()
        f[:, ny + 3:] = f[:, 3:6].clone()

    def bound_velocity(self, vel):
        nz = self.n[0]
        for c, f in enumerate(vel):
            self.wrap(f)
            if c == 2:
                f[2] = 0
                f[1], f[0] = -f[3], -f[4]
                f[nz + 2] = 0
                f[nz + 3], f[nz + 4] = -f[nz + 1], -f[nz]
                continue
            for j in range(3):
                f[2 - j] = -f[3 + j]  # no-slip floor
                f[nz + 3 + j] = -f[nz + 2 - j] if self.c.btype[capi.TO] == capi.NOSLIP else f[nz + 2]

    def bound_scalar(self, f):
        self.wrap(f)
        f[:3] = f[3].clone()
        f[self.n[0] + 3:] = f[self.n[0] + 2].clone()

    def subgrid(self):
        u, v, w = self.U
        a = self.at
        dx, dy, dz2 = self.dx, self.dy, 2 * self.dz2

        def cross(f, e, h):  # difference along h of f summed over the two faces o and e
            m = lambda s: [p + s * q for p, q in zip(e, h)]  # noqa: E731
            o = lambda s: [s * q for q in h]  # noqa: E731
            return a(f, *o(1)) + a(f, *m(1)) - a(f, *o(-1)) - a(f, *m(-1))

        X, Y, Z = (1, 0, 0), (0, 1, 0), (0, 0, 1)
        mx, my, mz = (-1, 0, 0), (0, -1, 0), (0, 0, -1)
        d00, d11 = (a(u) - a(u, -1)) / dx, (a(v) - a(v, 0, -1)) / dy
        d22 = (a(w) - a(w, 0, 0, -1)) / self.dzp
        s01 = (cross(u, mx, Y) / (4 * dy) + cross(v, my, X) / (4 * dx)) / 2
        s02 = (cross(u, mx, Z) / dz2 + cross(w, mz, X) / (4 * dx)) / 2
        s12 = (cross(v, my, Z) / dz2 + cross(w, mz, Y) / (4 * dy)) / 2
        s = d00 ** 2 + d11 ** 2 + d22 ** 2 + 2 * (s01 ** 2 + s02 ** 2 + s12 ** 2)
        width = (dx * dy * self.dzp) ** (1 / 3)
        f = torch.zeros_like(self.visc)
        self.at(f)[:] = torch.sqrt(2 * s) * (width * self.c.c_smag) ** 2 + self.c.nu
        self.wrap(f)
        f[2], f[self.n[0] + 3] = f[3], f[self.n[0] + 2]
        self.visc = f

    def at_point(self, c, p):
        """The velocity vector at the points p of component c."""
        out = []
        for d, f in enumerate(self.U):
            g, e, m = f.view(-1), self.pts.off[c], self.pts.off[d]
            out.append(g[p] if d == c else (g[p + e] + g[p] + g[p + e - m] + g[p - m]) / 4)
        return torch.stack(out, 1)

    def walls(self):
        """Momentum flux of every wall point, (tan / |tan|) u*^2, outwards."""
        self.stress = []
        for q, p, d, z0 in self.pts.wall:
            c = q // 6
            vel, dist = self.at_point(c, p), torch.linalg.vector_norm(d, dim=1)
            tan = vel - (vel * d).sum(1, keepdim=True) * d / (dist * dist)[:, None]
            mag = torch.linalg.vector_norm(tan, dim=1)
            old = self.ustar.get(q, torch.ones_like(mag))
            us = torch.where(z0 > 0, self.rough(mag, dist, z0), self.smooth(old, mag, dist))
            us = torch.where(mag != 0, us, old)
            self.ustar[q] = us
            t = torch.where(mag > math.sqrt(2.220446049250313e-16), tan[:, c] / mag * us * us, torch.zeros_like(mag))
            self.stress.append(t if q % 2 else -t)

    def rough(self, mag, dist, z0):
        lam = torch.sqrt(self.c.nu * mag / dist)
        log = mag * 0.41 / torch.log(dist / z0.clamp(min=1e-300))
        return torch.where(dist * lam / self.c.nu < 11.225 * 1.1, lam, log)

    def smooth(self, us, mag, dist):
        nu = self.c.nu
        lam = torch.sqrt(nu * mag / dist)
        done = dist * lam / nu < 5.0
        us = torch.where(done, lam, us)
        for _ in range(50):
            zpl = dist * us / nu
            lg = torch.log(zpl)
            new = torch.where(zpl <= 5, lam, torch.where(zpl < 30, mag / (5 * lg - float(np.float32(3.05))),
                                                         mag / (lg / 0.4 + 5.5)))
            new = torch.where(done, us, new)
            done, us = done | ((new - us).abs() / new.abs() < 1e-4), new
            if bool(done.all()):
                break
        return torch.where(done, us, torch.zeros_like(us))

    @staticmethod
    def shift(off, axis, m):
        r = list(off)
        r[axis] += m
        return r

    def advection4(self, c):
        """Fourth-order divergence form of component c."""
        f, o, acc = self.U[c], (0, 0, 0), 0.0
        for d, h in enumerate((self.dx, self.dy, self.c.dz)):
            def F(m):
                return self.at(f, *self.shift(o, d, m))

            def I(m):  # velocity d carried to the face m of f along d (times 16)
                if d == c:
                    g = lambda q: F(m + q)  # noqa: E731
                else:
                    g = lambda q: self.at(self.U[d], *self.shift(self.shift(o, d, m), c, q))  # noqa: E731
                return 9 * (g(0) + g(1)) - g(-1) - g(2)

            near = 9 * (I(0) * (F(0) + F(1)) - I(-1) * (F(-1) + F(0)))
            acc = acc + (near - (I(1) * (F(0) + F(3)) - I(-2) * (F(-3) + F(0))) / 3) / h
        return acc * (-1 / 256)

    def advection2(self, c, advective):
        """Second-order divergence form, or its mean with the advective form."""
        a, f, o, tot = self.at, self.U[c], (0, 0, 0), 0.0
        e = self.shift(o, c, 1)
        for d in range(3):
            p, m = self.shift(o, d, 1), self.shift(o, d, -1)
            g = self.U[d]
            if d == c:
                hi, lo, mid = a(f, *p) + a(f), a(f) + a(f, *m), 4 * a(f)
            else:
                me = [x + y for x, y in zip(m, e)]
                hi, lo = a(g, *e) + a(g), a(g, *me) + a(g, *m)
                mid = hi + lo
            h = (self.dx, self.dy, self.dzw if c == 2 else self.dzp)[d]
            h2 = (2 * self.dx, 2 * self.dy, self.dzw2 if c == 2 else self.dz2)[d]
            tot = tot - ((a(f, *p) + a(f)) * hi - (a(f) + a(f, *m)) * lo) / h / 4
            if advective:
                tot = tot - (a(f, *p) - a(f, *m)) / h2 * mid / 4
        return tot * 0.5 if advective else tot

    def advection(self, c):
        if self.vz:
            return self.advection2(c, True)
        t = self.at(self.pts.types[c])
        n = self.advection4(c)
        if bool((t != 0).any()):
            n = torch.where(t == 0, n, torch.where(t < 0, self.advection2(c, False), torch.zeros_like(n)))
        return n

    def diffusion(self, c):
        a, f, nu, o = self.at, self.U[c], self.visc, (0, 0, 0)
        tot, e = 0.0, self.shift(o, c, 1)
        for d, h in ((0, self.dx), (1, self.dy)):
            def flux(b):
                p = self.shift(b, d, 1)
                be, pe = ([x + y for x, y in zip(q, e)] for q in (b, p))
                v = a(nu, *p) if d == c else 0.25 * (a(nu, *pe) + a(nu, *be) + a(nu, *p) + a(nu, *b))
                return v * (a(f, *p) - a(f, *b)) / (h * h)

            tot = tot + flux(o) - flux(self.shift(o, d, -1))
        # faces 0..nz of the levels 1..nz
        L = lambda g, s=o: torch.cat([a(g, s[0], s[1], -1)[:1], a(g, s[0], s[1], 0)])  # noqa: E731
        H = lambda g, s=o: torch.cat([a(g, s[0], s[1], 0), a(g, s[0], s[1], 1)[-1:]])  # noqa: E731
        if c == 2:
            fz = H(nu) * (H(f) - L(f)) / self.dzu
        else:
            fz = 0.25 * (H(nu, e) + L(nu, e) + H(nu) + L(nu)) * (H(f) - L(f)) / self.dzf
        full = torch.zeros_like(f)
        a(full)[:] = tot + (fz[1:] - fz[:-1]) / (self.dzw if c == 2 else self.dzp)
        # at wall points the face's flux gives way to the wall stress
        off, g, m = self.pts.off, f.view(-1), nu.view(-1)
        for (q, p, _, _), stress in zip(self.pts.wall, self.stress):
            if q // 6 != c:
                continue
            d, plus = q % 6 // 2, q % 2
            b = p if plus else p - off[d]
            ee = off[c]
            v = m[b + off[d]] if d == c else 0.25 * (m[b + off[d] + ee] + m[b + ee] + m[b + off[d]] + m[b])
            far = b + off[d]
            k = b // off[2] - 2
            if d < 2:
                step = size = torch.full_like(stress, (self.dx, self.dy)[d])
                below = size
            else:
                step = (self.dzu if c == 2 else self.dzf).flatten()[k]
                sizes = (self.dzw if c == 2 else self.dzp).flatten()
                size, below = sizes[k.clamp(max=len(sizes) - 1)], sizes[(k - 1).clamp(min=0)]
            fl = v * (g[far] - g[b]) / step
            self.pts.add(full, far, (fl + stress) / size)
            self.pts.add(full, b, -(fl + stress) / below)
        return a(full)

    def scalar_tendency(self, s):
        a, f, o, eps = self.at, self.S[s], (0, 0, 0), float(np.float32(1e-8))
        t, pts, adv, dif = self.tdiff, self.pts, 0.0, 0.0
        for d, h in enumerate((self.dx, self.dy, self.c.dz)):
            def carried(b):
                u = a(self.U[d], *b)
                q = [a(f, *self.shift(b, d, m)) for m in (-1, 0, 1, 2)]
                up = u > 0
                sr = torch.where(up, q[2] - q[1], q[1] - q[2])
                sl = torch.where(up, q[1] - q[0], q[2] - q[3])
                sg = torch.copysign(torch.full_like(sl, eps), sl)
                r = (sr + sg) / (sl + sg)
                lim = torch.clamp(torch.minimum(2 * r, torch.clamp((1 + 2 * r) / 3, max=2.0)), min=0.0)
                return u * (torch.where(up, q[1], q[2]) + sl * lim / 2) * a(pts.open[d], *b) / h

            def spread(b):
                p = self.shift(b, d, 1)
                return (a(t, *p) + a(t, *b)) * (a(f, *p) - a(f, *b)) / (2 * h * h)

            m = self.shift(o, d, -1)
            adv = adv + carried(m) - carried(o)
            dif = dif + spread(o) - spread(m)
        full = torch.zeros_like(f)
        a(full)[:] = torch.where(a(pts.solid), torch.zeros_like(adv), adv) + dif
        g, tt = f.view(-1), t.view(-1)
        for d, h in enumerate((self.dx, self.dy, self.c.dz)):
            b, p = pts.faces[d], pts.faces[d] + pts.off[d]
            fl = (tt[p] + tt[b]) * (g[p] - g[b]) / (2 * h * h)
            pts.add(full, b, -fl)
            pts.add(full, p, fl)
        p, solid, div = pts.floor, pts.solid.view(-1), 0.0
        for d, h in enumerate((self.dx, self.dy, self.c.dz)):
            w, e = self.U[d].view(-1), pts.off[d]
            div = div + torch.where(solid[p + e], 0.0, w[p] / h) - torch.where(solid[p - e], 0.0, w[p - e] / h)
        pts.add(full, p, div * g[p])
        cell, which, amount = pts.src
        pts.add(full, cell[which == s], amount[which == s])
        return a(full)

    def project(self, vel, coef, mass):
        a, (nz, ny, nx) = self.at, self.n
        u, v, w = vel
        rhs = (a(u) - a(u, -1)) / self.dx + (a(v) - a(v, 0, -1)) / self.dy + (a(w) - a(w, 0, 0, -1)) / self.dzp
        x = torch.fft.rfft2((rhs if mass is None else rhs - a(mass)) / coef)

        def modes(m, n, h):
            return -4 * torch.sin(math.pi * torch.arange(m, device=_device(), dtype=torch.float64) / n) ** 2 / h ** 2

        lam = modes(ny, ny, self.dy)[:, None] + modes(nx // 2 + 1, nx, self.dx)[None]
        zw, zp = self.zw, self.zp
        low = [0.0] + [1 / ((zp[k] - zp[k - 1]) * (zw[k] - zw[k - 1])) for k in range(2, nz + 1)]
        up = [1 / ((zp[k + 1] - zp[k]) * (zw[k] - zw[k - 1])) for k in range(1, nz)] + [0.0]
        cp = []
        for k in range(nz):
            b = lam - low[k] - up[k]
            if k == 0:
                b[0, 0], x[0, 0, 0] = 1.0, 0.0  # the horizontal mean's level: x_1 = 0
                cp.append(up[0] / b)
                cp[0][0, 0] = 0.0
                x[0] /= b
                continue
            den = b - low[k] * cp[-1]
            cp.append(up[k] / den)
            x[k] = (x[k] - low[k] * x[k - 1]) / den
        for k in range(nz - 2, -1, -1):
            x[k] -= cp[k] * x[k + 1]
        phi = torch.fft.irfft2(x, s=(ny, nx))
        a(u)[:] -= coef / self.dx * (phi.roll(-1, 2) - phi)
        a(v)[:] -= coef / self.dy * (phi.roll(-1, 1) - phi)
        a(w)[:nz - 1] -= coef * (phi[1:] - phi[:-1]) / self.dzw[:nz - 1]
        p = a(self.P)
        p += phi
        p -= p[nz - 1].mean()
        self.wrap(self.P)

    def step(self):
        c, a, nz = self.c, self.at, self.n[0]
        u, v, w = self.U
        m = torch.maximum(a(u).abs(), a(u, -1).abs()) / self.dx + torch.maximum(a(v).abs(), a(v, 0, -1).abs()) / self.dy
        m = float((m + torch.maximum(a(w).abs(), a(w, 0, 0, -1).abs()) / self.dzp).max())
        self.dt = dt = min(c.cfl_target / m, c.dt_max) if c.variable_dt else c.dt
        self.cfl, self.time = m * dt, self.time + dt
        with_bodies = len(self.pts.taps[0][0]) > 0
        for st in range(3):
            rho, beta, coef = self.RHO[st] * dt, self.BETA[st] * dt, 2 * self.ALPHA[st] * dt
            self.subgrid()
            self.walls()
            self.pts.viscosity(self.visc)
            new = []
            for q in range(3):
                n = self.advection(q) + self.diffusion(q)
                f = rho * self.N[q] + beta * n
                self.N[q] = n
                if q == 0:
                    f = f - coef * c.pr_gradient_x
                h = (self.dx, self.dy, self.dzw)[q]
                f = f - coef * (a(self.P, *self.shift((0, 0, 0), q, 1)) - a(self.P)) / h
                if q == 2:
                    f[nz - 1] = 0
                g = self.U[q].clone()
                a(g)[:] += f
                new.append(g)
            for s in range(len(self.S)):
                n = self.scalar_tendency(s)
                f = self.S[s].clone()
                a(f)[:] += rho * self.NS[s] + beta * n
                self.NS[s] = n
                self.bound_scalar(f)
                self.S[s] = f
            mass = None
            self.bound_velocity(new)
            if with_bodies:
                self.pts.bodies(new)
                self.bound_velocity(new)
                mass = self.pts.mass(new, (c.dx, c.dy, c.dz))
            self.project(new, coef, mass)
            for f, p in zip(new, self.pts.null):
                f.view(-1)[p] = 0
            self.bound_velocity(new)
            if with_bodies:
                self.pts.bodies(new)
                self.bound_velocity(new)
            self.U = new


def _exact_fields(cfg, vel, lists, steps):
    f = _Flow(cfg, vel, lists)
    for _ in range(steps):
        f.step()
    out = dict(zip(("U", "V", "W", "Pr"), f.U + [f.P]))
    out.update({f"S{s}": g for s, g in enumerate(f.S)})
    return f, {name: f.at(g).contiguous().cpu().permute(2, 1, 0) for name, g in out.items()}


def _scenario(seed, cells, precision):
    cfg, cub, src, fields = serving.scenario(seed, cells, BITS[precision])
    vel = [torch.from_numpy(np.ascontiguousarray(f.T)).to(_device()) for f in fields[:3]]
    return cfg, vel, capi.Case(cfg, cuboids=cub, sources=src)


def exact(case, seed):
    """None for abl (iterated stability functions) and for runs of over about
    20 seconds."""
    if case["kind"] == "abl":
        return None
    if case["kind"] == "requests":
        out = {}
        for q, cells in enumerate(_request_cells(case)):
            _, got = _exact_fields(*_scenario(1000 * seed + q, cells, case["precision"]), case["steps"])
            out.update({f"{q}{name[0]}": v for name, v in got.items()})
        return out
    if case["kind"] == "scenario":
        return _exact_fields(*_scenario(seed, case["cells"], case["precision"]), case["steps"])[1]
    if case["nx"] * case["ny"] * case["nz"] * case["steps"] > 3e9:
        return None
    cfg = _config(case)
    cub, src = _bodies(case, seed)
    f, out = _exact_fields(cfg, _fields(case, seed)[0], capi.Case(cfg, cuboids=cub, sources=src), case["steps"])
    if case.get("diag"):
        out.update(cfl=f.cfl, dt=f.dt, time=f.time)
    return out
