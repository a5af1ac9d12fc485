"""The work that a user of life_amd has it do, as timed cases.

A pass is what a program does between two outputs: a number of time steps
(or a queue of served cases, or the layer-1 calls of a patched reference
solver) and the download of what it writes next -- density, velocity, marker
state and forces.  A case is a dict of plain values; ``prepare`` builds what
such a program holds, ``run`` does one pass through the public entry points,
``exact`` computes the same outputs in 64 bits with plain torch.

Kinds:
  cavity    lid-driven cavity, lattice only (walls on all sides)
  channel   inlet/outlet channel without bodies (pressure or convective outlet)
  cylinder  rigid cylinder in a channel: lattice + immersed boundary
  flag      inverted flag: one flexible filament, banded epsilon system
  plate     rigid cylinder with a flexible plate behind it, one epsilon system
  canopy    many flexible filaments on the bottom wall
  serve     a queue of independent flag cases through the serving engine
  layer1    the drop-in sequence of a patched reference solver: moving
            markers, supports, epsilon system, interpolation, spread
  transfer  restart-like use: a state is uploaded, advanced and downloaded
"""
import math
import random

import numpy as np
import torch

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case, Grid
from life_amd.serve import Server

PREC = {"f64": L.LIFE_FP64, "f32": L.LIFE_FP32_SHIFTED}


def listed():
    return [
        # the reference's LidDrivenCavity example grid: the smallest case it ships, latency-bound
        dict(name="cavity_101_cm_f64", kind="cavity", Nx=101, Ny=101, prec="f64", cm=True, steps=200),
        # the 256 x 256 BGK validation cavity
        dict(name="cavity_256_bgk_f32", kind="cavity", Nx=256, Ny=256, prec="f32", cm=False, steps=200),
        # a large wind-tunnel-like channel without bodies (the canopy's domain, half its sides)
        dict(name="channel_4096x2048_f32", kind="channel", Nx=4096, Ny=2048, prec="f32", cm=False, steps=100,
             outlet="convective"),
        # an ordinary plain-method channel of odd size, central moments
        dict(name="channel_1501x377_f64", kind="channel", Nx=1501, Ny=377, prec="f64", cm=True, steps=100,
             outlet="pressure"),
        # the reference's Cylinder example (Schaefer-Turek 2D-2), plain method
        dict(name="cylinder_441x83_f64", kind="cylinder", Nx=441, Ny=83, prec="f64", cm=False, steps=200,
             outlet="pressure"),
        # the 1024 x 256 validation cylinder, FP32-shifted, convective outlet
        dict(name="cylinder_1024x256_f32", kind="cylinder", Nx=1024, Ny=256, prec="f32", cm=True, steps=200,
             outlet="convective"),
        # the reference's InvertedFlag example grid, plain method (host FEM)
        dict(name="flag_631x451_f64", kind="flag", Nx=631, Ny=451, prec="f64", cm=False, steps=50, n_el=20),
        # the 2048 x 410 cylinder with a flexible plate, FP32-shifted (device FEM)
        dict(name="plate_2048x410_f32", kind="plate", Nx=2048, Ny=410, prec="f32", cm=True, steps=50, n_el=40),
        # the benchmark canopy: the largest case, 64 filaments
        dict(name="canopy_8192x4096_f32", kind="canopy", Nx=8192, Ny=4096, prec="f32", cm=False, steps=200,
             n_fil=64, L=200.0, n_el=50),
        # twelve cases of the serving stream's sizes, queued at once
        dict(name="serve_12_f32", kind="serve", n=12, prec="f32", cm=True, steps=60, wmax=2048, hmax=512),
        # a patched reference solver moving two filaments through the layer-1 calls
        dict(name="layer1_600x203_f64", kind="layer1", Nx=600, Ny=203, prec="f64", cm=False, steps=10, n_fil=2,
             L=81.0),
        # a restart-sized state in and out of the device around a few steps
        dict(name="transfer_1024x512_f64", kind="transfer", Nx=1024, Ny=512, prec="f64", cm=True, steps=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds; sizes over the listed ranges, odd ones among them."""
    kind = rng.choice(["cavity", "channel", "cylinder", "flag", "plate", "canopy", "serve", "layer1", "transfer"])
    prec = rng.choice(["f64", "f32"])
    cm = rng.random() < 0.5
    if kind == "cavity":
        return dict(kind=kind, Nx=_log(rng, 40, 2100), Ny=_log(rng, 40, 2100), prec=prec, cm=cm,
                    steps=rng.randint(50, 200))
    if kind == "channel":
        return dict(kind=kind, Nx=_log(rng, 300, 4096), Ny=_log(rng, 50, 2048), prec=prec, cm=cm,
                    steps=rng.randint(40, 100), outlet=rng.choice(["pressure", "convective"]))
    if kind == "cylinder":
        Ny = _log(rng, 83, 420)
        return dict(kind=kind, Nx=int(Ny * rng.uniform(3.5, 5.5)), Ny=Ny, prec=prec, cm=cm,
                    steps=rng.randint(50, 200), outlet=rng.choice(["pressure", "convective"]))
    if kind == "flag":
        Ny = _log(rng, 128, 512)
        return dict(kind=kind, Nx=int(Ny * rng.uniform(1.4, 4.0)), Ny=Ny, prec=prec, cm=True,
                    steps=rng.randint(20, 50), n_el=rng.randint(20, 60))
    if kind == "plate":
        Ny = _log(rng, 150, 410)
        return dict(kind=kind, Nx=5 * Ny, Ny=Ny, prec=prec, cm=True, steps=rng.randint(20, 50),
                    n_el=rng.randint(20, 40))
    if kind == "canopy":
        n = rng.randint(4, 32)
        return dict(kind=kind, Nx=_log(rng, 2400, 8192), Ny=_log(rng, 400, 2048), prec=prec, cm=False,
                    steps=rng.randint(20, 60), n_fil=n, L=float(rng.randint(60, 200)), n_el=rng.randint(20, 50))
    if kind == "serve":
        return dict(kind=kind, n=rng.randint(3, 12), prec=prec, cm=True, steps=rng.randint(20, 60),
                    wmax=rng.choice([1024, 2048]), hmax=rng.choice([256, 512]))
    if kind == "layer1":
        return dict(kind=kind, Nx=_log(rng, 240, 1200), Ny=_log(rng, 96, 300), prec=prec, cm=cm,
                    steps=rng.randint(4, 12), n_fil=rng.randint(1, 3), L=float(rng.randint(24, 60)))
    return dict(kind=kind, Nx=_log(rng, 100, 2048), Ny=_log(rng, 60, 1024), prec=prec, cm=cm, steps=rng.randint(1, 20))


# ---------------------------------------------------------------- inputs

def _setup(case, seed):
    """(CaseParams, geometry text) of a simulated case; the seed moves speeds,
    viscosities and positions by a few per cent."""
    rng = random.Random("%d %s" % (seed, case["kind"]))
    s = rng.uniform(0.9, 1.1)
    r = rng.uniform(0.9, 1.1)
    Nx, Ny, cm, kind = case["Nx"], case["Ny"], int(case["cm"]), case["kind"]
    if kind == "cavity":
        p, g = cfg.lid_driven_cavity(N=Ny, tau=0.5 + 0.1 * r, u_lid=0.05 * s, central_moments=cm)
        return p.replace(Nx=Nx), g
    if kind in ("channel", "transfer"):
        right = cfg.CONVECTIVE if case.get("outlet") == "convective" else cfg.PRESSURE
        p = cfg.lattice_case(Nx, Ny, 0.5 + 0.08 * r, wall_left=cfg.VELOCITY, wall_right=right, wall_bottom=cfg.WALL,
                             wall_top=cfg.FREESLIP, profile=cfg.BOUNDARY_LAYER, uxInlet_p=0.04 * s,
                             central_moments=cm)
        return p, ""
    if kind == "cylinder":
        D = 0.16 * (Ny - 1)
        right = cfg.CONVECTIVE if case["outlet"] == "convective" else cfg.PRESSURE
        p, g = cfg.cylinder_channel(Nx=Nx, Ny=Ny, D=D, u_max=0.04 * s, Re=80.0 * r, ramp_steps=0.0,
                                    centre=(0.22 * Nx + rng.uniform(-0.5, 0.5), 0.49 * Ny + rng.uniform(-0.5, 0.5)))
        return p.replace(central_moments=cm, wall_right=right), g
    if kind == "flag":
        p, g = cfg.inverted_flag(Nx, Ny, 0.2, case["n_el"], Re=100.0 * r, kb=0.8 * s, central_moments=cm,
                                 u_in=0.04)
        return p, g
    if kind == "plate":
        D = 0.195 * Ny
        p, g = cfg.flexible_fsi(Nx=Nx, Ny=Ny, D=D, centre=(0.5 * Ny, 0.488 * Ny), L=3.5 * D, h=0.2 * D,
                                n_el=case["n_el"], u_mean=0.03 * s, Re=100.0 * r, ramp_steps=0.0,
                                central_moments=cm)
        return p, g
    if kind in ("canopy", "layer1"):
        Lf = case["L"]
        if kind == "canopy":
            gap, box = min(60.0, 0.4 * Nx / case["n_fil"]), None
        else:
            gap, box = 0.15 * Nx, (0.2 * Nx, 0.7 * Nx)
        p, g = cfg.canopy(Nx=Nx, Ny=Ny, n_filaments=case["n_fil"], L=Lf, n_el=case.get("n_el", 10), min_spacing=gap,
                          u_in=0.05 * s, seed=rng.randrange(1 << 30), ramp_steps=0.0, x_range=box,
                          kb_range=(0.1, 1.0))
        return p.replace(ux0_p=0.05 * s, central_moments=cm), g
    raise KeyError(kind)


def _requests(case, seed):
    """The case's queue: sizes and element counts as the serving stream draws
    them (the same for every seed), Reynolds number, stiffness and inflow from
    the seed."""
    heights = [h for h in (128, 256, 512) if h <= case["hmax"]]
    widths = [w for w in (512, 1024, 2048) if w <= case["wmax"]]
    sizes, rng = random.Random(case["n"]), random.Random(seed)
    out = []
    for _ in range(case["n"]):
        Nx, Ny, n_el = sizes.choice(widths), sizes.choice(heights), sizes.randint(20, 60)
        kb = math.exp(rng.uniform(math.log(0.2), 0.0))
        p, g = cfg.inverted_flag(Nx, Ny, 0.25, n_el, Re=rng.uniform(50.0, 200.0), kb=kb, central_moments=1,
                                 u_in=0.04 * rng.uniform(0.9, 1.1))
        out.append(dict(params=p, geometry=g, steps=case["steps"]))
    return out


def _filaments(case, geometry):
    """Markers of the canopy's vertical filaments one lattice spacing apart: positions, body index, roots."""
    pos, body, roots = [], [], []
    for b, line in enumerate(geometry.strip().splitlines()):
        x = float(line.split()[3])
        n = int(case["L"]) + 1
        pos += [(x, float(k)) for k in range(n)]
        body += [b] * n
        roots.append(x)
    return np.array(pos), np.array(body, dtype=np.int32), roots


def _bend(case, pos0, t):
    """Prescribed bending of the filaments at time t (clamped at the wall): positions and velocities."""
    s = pos0[:, 1] / case["L"]
    w = 2.0 * math.pi / 100.0
    pos, vel = pos0.copy(), np.zeros_like(pos0)
    pos[:, 0] += 1.5 * math.sin(w * t) * s * s
    vel[:, 0] = 1.5 * w * math.cos(w * t) * s * s
    return pos, vel


def _state_arrays(case, seed):
    """A smooth flow with noise and its populations (a restart file's content)."""
    rng = np.random.default_rng(seed)
    Nx, Ny = case["Nx"], case["Ny"]
    x = np.linspace(0.0, 2.0 * math.pi, Nx)[:, None]
    y = np.linspace(0.0, 2.0 * math.pi, Ny)[None, :]
    rho = 1.0 + 0.01 * np.sin(x + seed % 7) * np.cos(y) + 1e-3 * rng.standard_normal((Nx, Ny))
    u = np.stack([0.04 * np.sin(y) * np.cos(x), 0.03 * np.sin(x) * np.ones_like(y)], axis=-1)
    u += 1e-3 * rng.standard_normal((Nx, Ny, 2))
    f = np.empty((Nx, Ny, 9))
    uu = 1.5 * (u[..., 0] ** 2 + u[..., 1] ** 2)
    for v in range(9):
        cu = 3.0 * (CX[v] * u[..., 0] + CY[v] * u[..., 1])
        f[..., v] = W[v] * rho * (1.0 + cu + 0.5 * cu * cu - uu)
    f *= 1.0 + 1e-3 * rng.standard_normal((Nx, Ny, 9))
    return f, rho, u


def prepare(case, seed):
    prec = PREC[case["prec"]]
    if case["kind"] == "serve":
        srv = Server(precision=prec, max_cases=16)
        return dict(kind="serve", server=srv, stream=_requests(case, seed))
    p, g = _setup(case, seed)
    if case["kind"] == "transfer":
        f, rho, u = _state_arrays(case, seed)
        return dict(kind="transfer", case=case, grid=Grid(p, precision=prec), f=f, rho=rho, u=u)
    if case["kind"] == "layer1":
        pos0, body, roots = _filaments(case, g)
        gr = Grid(p, precision=prec)
        gr.set_markers(pos0, np.zeros_like(pos0), body, [0] * len(roots))
        return dict(kind="layer1", case=case, grid=gr, pos0=pos0, body=body, nb=len(roots), t=0)
    # the output buffers that a program keeps between its outputs
    out = dict(rho=np.zeros((case["Nx"], case["Ny"])), u=np.zeros((case["Nx"], case["Ny"], 2)))
    return dict(kind=case["kind"], case=case, sim=Case(p, g, precision=prec), out=out)


# ---------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "serve":
        return _run_serve(state)
    if kind == "transfer":
        return _run_transfer(state)
    if kind == "layer1":
        return _run_layer1(state)
    sim, out = state["sim"], state["out"]
    sim.step(state["case"]["steps"])
    L.check(L.load().life_grid_download(sim.grid.h, None, L.dptr(out["rho"]), L.dptr(out["u"]), None))
    if sim.n_markers:
        m = sim.markers()
        for k in ("pos", "vel", "force", "eps"):
            out[k] = m[k]
        out["total_force"] = sim.total_force()
        flex = [b for b in range(sim.n_bodies) if sim.body_info(b)["flex"] == 0]
        if flex:
            out["fem_U"] = np.concatenate([sim.fem(b)[0] for b in flex])
    return out


def _run_serve(state):
    srv = state["server"]
    ids = [srv.submit(r["params"], r["geometry"], r["steps"], keep_fields=True) for r in state["stream"]]
    srv.drain()
    out = {}
    for k, rid in enumerate(ids):
        info = srv.info(rid)
        if info["status"] != L.LIFE_REQ_DONE:
            raise RuntimeError(srv.error(rid))
        rho, u, pos = srv.fields(rid)
        out["case%02d" % k] = dict(rho=rho, u=u, pos=pos, force=np.array(info["total_force"] + info["tip"]))
        srv.release(rid)
    return out


def _run_transfer(state):
    gr = state["grid"]
    gr.upload(state["f"], state["rho"], state["u"])
    for t in range(1, state["case"]["steps"] + 1):
        gr.lbm_kernel(t)
    f, rho, u, _ = gr.download()
    return dict(f=f, rho=rho, u=u)


def _run_layer1(state):
    gr, case = state["grid"], state["case"]
    n = len(state["pos0"])
    m = n // state["nb"]
    for _ in range(case["steps"]):
        state["t"] += 1
        gr.lbm_kernel(state["t"])
        pos, vel = _bend(case, state["pos0"], state["t"])
        gr.update_markers(pos, vel)
        gr.find_support(1)
        eps = np.zeros(n)
        for b in range(state["nb"]):
            A = gr.epsilon_matrix(b * m, m)
            eps[b * m:(b + 1) * m] = L.solve_lapack(A, np.ones(m))
        gr.set_epsilon(eps)
        force = gr.interpolate()
        gr.spread()
    _, rho, u, fibm = gr.download()
    mk = gr.markers()
    return dict(rho=rho, u=u, fibm=fibm, A=A, force=force, eps=mk["eps"], ds=mk["ds"], supp=mk["supp_ij"],
                delta=mk["supp_delta"])


# ---------------------------------------------------------------- work

def work(case):
    """Bytes: a pass reads the populations and writes them once (what lies
    between the steps of a pass may stay on the chip), and writes its outputs
    once.  Flops: about 250 a site update for BGK, 450 for central moments."""
    pop = 4.0 if case["prec"] == "f32" else 8.0
    per = 450.0 if case["cm"] else 250.0
    if case["kind"] == "serve":
        # mean lattice of the stream
        w = [x for x in (512, 1024, 2048) if x <= case["wmax"]]
        h = [x for x in (128, 256, 512) if x <= case["hmax"]]
        N = case["n"] * (sum(w) / len(w)) * (sum(h) / len(h))
    else:
        N = float(case["Nx"] * case["Ny"])
    S = case["steps"]
    out = {"transfer": (9 + 3 + 9 + 3) * 8.0, "layer1": 5 * 8.0}.get(case["kind"], 3 * 8.0)
    return {"bytes": N * (18.0 * pop + out), "flops": N * S * per}


# ---------------------------------------------------------------- 64-bit values without life_amd's kernels

CX = (0, 1, -1, 0, 0, 1, -1, 1, -1)
CY = (0, 0, 0, 1, -1, 1, -1, -1, 1)
W = (4 / 9,) + (1 / 9,) * 4 + (1 / 36,) * 4
OPP = (0, 2, 1, 4, 3, 6, 5, 8, 7)
D = torch.float64


def exact(case, seed):
    """The lattice method with its boundary conditions, and the immersed
    boundary for rigid or prescribed bodies.  A flexible body's Newmark /
    corotational beam iteration has no plain restatement here: None."""
    kind = case["kind"]
    if kind in ("flag", "plate", "canopy", "serve"):
        return None
    p, g = _setup(case, seed)
    S = case["steps"]
    lat = _Lattice(p)
    if kind == "transfer":
        f, rho, u = _state_arrays(case, seed)
        lat.load(f, rho, u)
    if kind == "cylinder":
        lat.circle(g)
    if kind == "layer1":
        pos0, body, roots = _filaments(case, g)
    for t in range(1, S + 1):
        lat.step(t)
        if kind == "cylinder":
            lat.couple()
        elif kind == "layer1":
            lat.move(*_bend(case, pos0, t), body)
            lat.couple()
    out = dict(rho=lat.rho.cpu(), u=lat.u.permute(1, 2, 0).cpu())
    if kind == "transfer":
        out["f"] = lat.f.permute(1, 2, 0).cpu()
    elif kind == "cylinder":
        out.update(pos=lat.pos.cpu(), vel=lat.vel.cpu(), force=lat.force.cpu(), eps=lat.eps.cpu(),
                   total_force=lat.total_force().cpu())
    elif kind == "layer1":
        out.update(fibm=lat.fibm.permute(1, 2, 0).cpu(), A=lat.A.cpu(), force=lat.force.cpu(), eps=lat.eps.cpu(),
                   ds=lat.ds.cpu(), supp=None, delta=None)
    return out


class _Lattice:
    """D2Q9 step on whole planes f[v, i, j], with regularised boundaries."""

    def __init__(self, p):
        self.p = p
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.cx = torch.tensor(CX, dtype=D, device=self.dev).view(9, 1, 1)
        self.cy = torch.tensor(CY, dtype=D, device=self.dev).view(9, 1, 1)
        self.w = torch.tensor(W, dtype=D, device=self.dev).view(9, 1, 1)
        h = p.height_p / (p.Ny - 1)
        self.omega = p.omega if p.omega > 0 else 1.0 / (3.0 * p.nu_p * p.tStep / (h * h) + 0.5)
        nu = (1.0 / self.omega - 0.5) / 3.0
        self.Dx, self.Dt = h, h * h * nu / p.nu_p
        self.Dm = p.rho_p * h ** 3
        y = torch.arange(p.Ny, dtype=D, device=self.dev) * h
        U = torch.tensor([p.uxInlet_p, p.uyInlet_p], dtype=D, device=self.dev).view(2, 1) * self.Dt / h
        H = p.height_p
        shape = {cfg.UNIFORM: torch.ones_like(y), cfg.PARABOLIC: 1.5 * (1 - ((y - H / 2) / (H / 2)) ** 2),
                 cfg.SHEAR: y / H, cfg.BOUNDARY_LAYER: 1.5 * y * (2 * H - y) / (H * H)}[p.profile]
        self.uin = U * shape
        self.rho = torch.ones(p.Nx, p.Ny, dtype=D, device=self.dev)
        if p.profile != cfg.UNIFORM:
            self.u = self.uin.view(2, 1, p.Ny).repeat(1, p.Nx, 1)
        else:
            u0 = torch.tensor([p.ux0_p, p.uy0_p], dtype=D, device=self.dev) * self.Dt / h
            self.u = u0.view(2, 1, 1).repeat(1, p.Nx, p.Ny)
        self.groups, self.conv = self._boundaries()
        for key, (i, j) in self.groups.items():
            if key[0] == cfg.WALL:
                self.u[:, i, j] = 0.0
        self.f = self.feq(self.rho, self.u)
        self.fibm = torch.zeros_like(self.u)

    def load(self, f, rho, u):
        self.f = torch.tensor(f, device=self.dev).permute(2, 0, 1).contiguous()
        self.rho = torch.tensor(rho, device=self.dev)
        self.u = torch.tensor(u, device=self.dev).permute(2, 0, 1).contiguous()

    def _type(self, i, j):
        p = self.p
        if j == 0:
            return p.wall_bottom
        if j == p.Ny - 1:
            return p.wall_top
        return p.wall_left if i == 0 else p.wall_right if i == p.Nx - 1 else cfg.FLUID

    def _boundaries(self):
        p, groups, conv = self.p, {}, []
        edge = [(i, j) for i in (0, p.Nx - 1) for j in range(p.Ny)]
        edge += [(i, j) for i in range(1, p.Nx - 1) for j in (0, p.Ny - 1)]
        for i, j in edge:
            t = self._type(i, j)
            if t == cfg.FLUID:
                continue
            if t == cfg.CONVECTIVE:
                conv.append(j)
                continue
            nx = 1 if i == 0 else -1 if i == p.Nx - 1 else 0
            ny = 1 if j == 0 else -1 if j == p.Ny - 1 else 0
            if nx and ny:  # a corner beside an open side takes the other side's normal
                if self._type(i + nx, j) == cfg.FLUID:
                    ny = 0
                elif self._type(i, j + ny) == cfg.FLUID:
                    nx = 0
            groups.setdefault((t, nx, ny), []).append((i, j))
        idx = {k: tuple(torch.tensor(c, device=self.dev) for c in zip(*v)) for k, v in groups.items()}
        return idx, torch.tensor(conv, dtype=torch.long, device=self.dev)

    def feq(self, rho, u):
        cx, cy, w = (a.view([9] + [1] * rho.dim()) for a in (self.cx, self.cy, self.w))
        x, y = u[0], u[1]
        if self.p.central_moments:
            ax = 9 * cx * cx * x * x + 6 * cx * x - 3 * x * x + 2
            ay = 9 * cy * cy * y * y + 6 * cy * y - 3 * y * y + 2
            return 0.25 * rho * w * ax * ay
        cu = cx * x + cy * y
        return rho * w * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * (x * x + y * y))

    def collide(self):
        p, f, rho, u, F = self.p, self.f, self.rho, self.u, self.fibm
        om = self.omega
        if not p.central_moments:
            cu = self.cx * u[0] + self.cy * u[1]
            guo = 3 * self.w * (F[0] * (self.cx - u[0] + 3 * self.cx * cu) + F[1] * (self.cy - u[1] + 3 * self.cy * cu))
            return f + om * (self.feq(rho, u) - f) + (1 - 0.5 * om) * guo
        # central moments: the two second-order shear moments relax, the
        # others take their equilibrium (plus the force)
        dx, dy = self.cx - u[0], self.cy - u[1]
        k4 = (1 - om) * (f * (dx * dx - dy * dy)).sum(0)
        k5 = (1 - om) * (f * dx * dy).sum(0)
        k3 = 2 * rho / 3
        fx, fy = 0.5 * F[0], 0.5 * F[1]
        n = [[rho, fy, 0.5 * (k3 - k4)], [fx, k5, fx / 3], [0.5 * (k3 + k4), fy / 3, rho / 9]]  # [x power][y power]
        for a in range(3):
            n[a] = self._pops(n[a], u[1])
        cols = [self._pops([n[a][b] for a in range(3)], u[0]) for b in range(3)]  # cols[cy][cx], order 0, 1, -1
        return torch.stack([cols[CY[v]][CX[v]] for v in range(9)])

    @staticmethod
    def _pops(n, u):
        """Central moments of order 0..2 about u along one axis to the values at c = 0, 1, -1."""
        m1 = n[1] + u * n[0]
        m2 = n[2] + 2 * u * n[1] + u * u * n[0]
        return [n[0] - m2, 0.5 * (m2 + m1), 0.5 * (m2 - m1)]

    def step(self, t):
        p = self.p
        ramp = 1.0
        if p.inlet_ramp > 0 and self.Dt * t <= p.inlet_ramp:
            ramp = 0.5 * (1 - math.cos(math.pi * self.Dt * t / p.inlet_ramp))
        u1, u2, u3 = self.u[:, -1], self.u[:, -2], self.u[:, -3]
        delU = -0.5 * u1[0].mean() * (3 * u1 - 4 * u2 + u3)
        post = self.collide()
        new = torch.empty_like(post)
        for v in range(9):
            new[v] = torch.roll(post[v], (CX[v], CY[v]), (0, 1))
        if len(self.conv):
            j = self.conv
            for v in (2, 6, 8):
                new[v, -1, j] = self.f[v, -1, j] + 3 * W[v] * (delU[0, j] * CX[v] + delU[1, j] * CY[v])
        self.f = new
        self._walls(ramp)
        self.rho = self.f.sum(0)
        self.mom = torch.stack([(self.cx * self.f).sum(0), (self.cy * self.f).sum(0)])
        self.u = self.mom / self.rho
        self.fibm = torch.zeros_like(self.u)

    def _walls(self, ramp):
        done = []
        for (typ, nx, ny), (i, j) in self.groups.items():
            f = self.f[:, i, j].clone()
            n1, n2 = self.f[:, i + nx, j + ny], self.f[:, i + 2 * nx, j + 2 * ny]
            u = torch.zeros(2, len(i), dtype=D, device=self.dev)
            c = CX if nx else CY
            s = nx if nx else ny
            if typ == cfg.VELOCITY:
                u = self.uin[:, j] * ramp
            elif typ in (cfg.FREESLIP, cfg.PRESSURE):
                cx, cy = self.cx.view(9, 1), self.cy.view(9, 1)
                for d, cc in enumerate((cx, cy)):
                    if (d == 0) == (not nx):  # along the side (both at a corner: neither)
                        g1 = (cc * n1).sum(0) / n1.sum(0)
                        g2 = (cc * n2).sum(0) / n2.sum(0)
                        if not (nx and ny):
                            u[d] = (4 * g1 - g2) / 3
            if nx and ny:
                if typ in (cfg.FREESLIP, cfg.PRESSURE):
                    u = self._corner_slip(n1, n2, nx, ny)
                rho = 2 * n1.sum(0) - n2.sum(0)
            else:
                out = sum(f[v] for v in range(9) if c[v] == -s)
                zero = sum(f[v] for v in range(9) if c[v] == 0)
                d = 0 if nx else 1
                if typ == cfg.PRESSURE:
                    rho = torch.ones(len(i), dtype=D, device=self.dev)
                    u[d] = s * (1 - (2 * out + zero) / rho)
                else:
                    rho = (2 * out + zero) / (1 - s * u[d])
            eq = self.feq(rho, u)
            neq = f - eq
            for v in range(9):
                unknown = (CX[v] == nx or CY[v] == ny) if nx and ny else c[v] == s
                if unknown:
                    buried = nx and ny and nx * CX[v] + ny * CY[v] == 0
                    neq[v] = torch.zeros_like(rho) if buried else f[OPP[v]] - eq[OPP[v]]
            sxx = sum(CX[v] * CX[v] * neq[v] for v in range(9))
            syy = sum(CY[v] * CY[v] * neq[v] for v in range(9))
            sxy = sum(CX[v] * CY[v] * neq[v] for v in range(9))
            reg = torch.stack([eq[v] + 4.5 * W[v] * ((CX[v] ** 2 - 1 / 3) * sxx + (CY[v] ** 2 - 1 / 3) * syy +
                                                     2 * CX[v] * CY[v] * sxy) for v in range(9)])
            done.append((i, j, reg))
        for i, j, reg in done:
            self.f[:, i, j] = reg

    def _corner_slip(self, n1, n2, nx, ny):
        """Free-slip corner: its side is the bottom or top, so the normal
        velocity is zero and the tangential one has zero gradient."""
        cx = self.cx.view(9, 1)
        u = torch.zeros(2, n1.shape[1], dtype=D, device=self.dev)
        u[0] = (4 * (cx * n1).sum(0) / n1.sum(0) - (cx * n2).sum(0) / n2.sum(0)) / 3
        return u

    # -- immersed boundary
    def circle(self, geometry):
        x, y, r = (float(geometry.split()[k]) for k in (3, 4, 7))
        n = int(math.floor(2 * math.pi * r / self.Dx))
        a = torch.arange(n, dtype=D, device=self.dev) * 2 * math.pi / n
        pos = torch.stack([x + r * torch.cos(a), y + r * torch.sin(a)], 1)
        self.move(pos, torch.zeros_like(pos), np.zeros(n, dtype=np.int32))

    @staticmethod
    def _delta(r):
        a = r.abs()
        inner = (1 + torch.sqrt((1 - 3 * a * a).clamp(min=0))) / 3
        outer = (5 - 3 * a - torch.sqrt((1 - 3 * (1 - a) ** 2).clamp(min=0))) / 6
        return torch.where(a <= 0.5, inner, torch.where(a <= 1.5, outer, torch.zeros_like(a)))

    def move(self, pos, vel, body):
        self.pos = torch.as_tensor(pos, dtype=D, device=self.dev)
        self.vel = torch.as_tensor(vel, dtype=D, device=self.dev)
        body = torch.as_tensor(np.asarray(body), device=self.dev)
        x = self.pos / self.Dx
        base = torch.floor(x + 0.5)
        off = torch.arange(-2, 3, dtype=D, device=self.dev)
        si = base[:, 0, None] + off
        sj = base[:, 1, None] + off
        dx, dy = (x[:, 0, None] - si).abs(), (x[:, 1, None] - sj).abs()
        okx = (dx < 1.5) & (si >= 0) & (si <= self.p.Nx - 1)
        oky = (dy < 1.5) & (sj >= 0) & (sj <= self.p.Ny - 1)
        self.wx = torch.where(okx, self._delta(dx), torch.zeros_like(dx))
        self.wy = torch.where(oky, self._delta(dy), torch.zeros_like(dy))
        self.si, self.sj = si, sj
        self.ii = si.clamp(0, self.p.Nx - 1).long()
        self.jj = sj.clamp(0, self.p.Ny - 1).long()
        diff = self.pos[:, None] - self.pos[None]
        d = diff.pow(2).sum(-1).sqrt() / self.Dx
        other = (body[:, None] != body[None]) | torch.eye(len(d), dtype=torch.bool, device=self.dev)
        self.ds = torch.where(other, torch.full_like(d, 10.0), d).amin(1).clamp(max=10.0)
        # A_ij = sum over the supports s of i of delta_i(s) delta(x_j - s), times ds_j
        ax = torch.einsum("ia,ija->ij", self.wx, self._delta(x[None, :, 0, None] - si[:, None]))
        ay = torch.einsum("ia,ija->ij", self.wy, self._delta(x[None, :, 1, None] - sj[:, None]))
        A = ax * ay * self.ds
        self.eps = torch.zeros(len(d), dtype=D, device=self.dev)
        for b in body.unique():
            k = torch.nonzero(body == b).flatten()
            self.A = A[k][:, k]
            self.eps[k] = torch.linalg.solve(self.A.cpu(), torch.ones(len(k), dtype=D)).to(self.dev)

    def couple(self):
        w = self.wx[:, :, None] * self.wy[:, None, :]
        i = self.ii[:, :, None].expand_as(w)
        j = self.jj[:, None, :].expand_as(w)
        rho = (w * self.rho[i, j]).sum((1, 2))
        mom = torch.stack([(w * self.mom[d][i, j]).sum((1, 2)) for d in (0, 1)], 1)
        self.force = 2 * (self.Dt / self.Dx * rho[:, None] * self.vel - mom)
        s = self.eps * self.ds
        for d in (0, 1):
            self.fibm[d].index_put_((i.reshape(-1), j.reshape(-1)),
                                    ((self.force[:, d] * s)[:, None, None] * w).reshape(-1), accumulate=True)
        self.u = (self.mom + 0.5 * self.fibm) / self.rho

    def total_force(self):
        F = -(self.force * (self.eps * self.ds)[:, None]).sum(0) * self.Dm / (self.Dt * self.Dt)
        return torch.cat([F, F / (0.5 * self.p.ref_rho * self.p.ref_U ** 2 * self.p.ref_L)])
