"""The tiled step (several steps of a lattice without bodies in one launch)
against the plain kernels and the oracle.

Sizes: one tile spanning the lattice, tiles that divide it unevenly, thin
lattices whose tiles touch both walls, every default tile shape (8, 12, 16,
20, 24 squares; the 16 x 32 blocks of larger lattices); step counts that leave
1, 2 and 3 steps for the last launch.  The tiled step does the plain kernels'
operations on the same operands: results equal bit for bit, in FP64 and FP32.
"""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case
from tests._util import bc_mix_params, rel_err

pytestmark = pytest.mark.gpu

SIZES = [(4, 4), (5, 9), (40, 24), (9, 300), (200, 187), (260, 251), (310, 301), (370, 381), (700, 6), (530, 420)]


def params(kind, Nx, Ny, cm):
    if kind == "periodic":
        return cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.FLUID, wall_right=cfg.FLUID, wall_bottom=cfg.FLUID,
                                wall_top=cfg.FLUID, profile=cfg.UNIFORM, uxInlet_p=0.0, ux0_p=0.03, dpdx=1e-5,
                                central_moments=cm)
    if kind == "womersley":
        return cfg.womersley_channel(Nx=Nx, Ny=Ny, central_moments=cm)
    return bc_mix_params(kind, Nx=Nx, Ny=Ny, cm=cm)[0]


def fields(p, prec, steps, state=None):
    c = Case(p, "", precision=prec)
    if state is not None:
        c.grid.upload(*state)
    for n in steps:
        c.step(n)
    out = c.fields()
    c.close()
    return out


@pytest.mark.parametrize("cm", [0, 1])
@pytest.mark.parametrize("kind", ["ldc", "channel_pressure", "periodic_force", "boundary_layer", "periodic", "womersley"])
def test_tiled_step_equals_plain_kernels(gpu_lib, monkeypatch, kind, cm):
    for Nx, Ny in SIZES:
        p = params(kind, Nx, Ny, cm)
        rng = np.random.default_rng(Nx + Ny)
        w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
        f = w * (1.0 + 0.02 * rng.standard_normal((Nx, Ny, 9)))
        state = (f, f.sum(-1), 0.01 * rng.standard_normal((Nx, Ny, 2)))
        for prec in (L.LIFE_FP64, L.LIFE_FP32_SHIFTED):
            monkeypatch.delenv("LIFE_TILE", raising=False)
            tiled = fields(p, prec, (1, 9, 2), state)
            monkeypatch.setenv("LIFE_TILE", "0")
            plain = fields(p, prec, (1, 9, 2), state)
            assert np.isfinite(plain[0]).all()
            for a, b in zip(tiled, plain):
                assert np.array_equal(a, b), (kind, cm, Nx, Ny, prec, float(np.abs(a - b).max()))


@pytest.mark.parametrize("kind", ["ldc", "channel_pressure", "periodic_force"])
def test_tiled_step_matches_oracle(oracle, gpu_lib, kind):
    p = params(kind, 101, 63, 1)
    oc = oracle.OracleCase(p, "")
    oc.step(31)
    f, rho, u, _ = fields(p, L.LIFE_FP64, (31,))
    fo, ro, uo, _ = oc.grid()
    assert max(rel_err(f, fo), rel_err(rho, ro), rel_err(u, uo)) <= 1e-12
    oc.close()


def test_blow_up_is_reported_at_its_scan(gpu_lib, monkeypatch):
    """A NaN is found at the same scan (every 10 steps) and site as by the plain kernels."""
    p = params("ldc", 60, 50, 0)
    msg = []
    for tile in (None, "0"):
        monkeypatch.delenv("LIFE_TILE", raising=False)
        if tile:
            monkeypatch.setenv("LIFE_TILE", tile)
        c = Case(p, "", precision=L.LIFE_FP64)
        c.set_check_interval(10)
        c.step(5)
        f, rho, u, _ = c.fields()
        f[20, 30, 0] = np.nan
        c.grid.upload(f, rho, u)
        with pytest.raises(L.LifeError) as e:
            c.step(40)
        msg.append(str(e.value))
        c.close()
    assert msg[0] == msg[1] and "t = 10)" in msg[0]


def one_step_cases(cm):
    cyl, g = cfg.cylinder_channel(Nx=241, Ny=61, D=10.0, u_max=0.05, Re=60.0, ramp_steps=0.0, centre=(60.2, 29.7))
    yield "cylinder, convective", cyl.replace(central_moments=cm), g
    yield "cylinder, pressure", cyl.replace(central_moments=cm, wall_right=cfg.PRESSURE), g
    # larger tiles; body two columns from the outlet, so that its supports carry force in the outlet's three columns
    p, g = cfg.cylinder_channel(Nx=410, Ny=391, D=40.0, u_max=0.05, Re=60.0, ramp_steps=0.0, centre=(387.3, 190.2))
    yield "cylinder at the outlet", p.replace(central_moments=cm), g
    # more outlet rows than threads of the outlet mean
    yield "tall channel", bc_mix_params("channel_convective", Nx=60, Ny=1100, cm=cm)[0], ""
    yield "thin channel", bc_mix_params("channel_convective", Nx=6, Ny=5, cm=cm)[0], ""
    yield "pressure corners", cfg.lattice_case(50, 33, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE,
                                               wall_bottom=cfg.PRESSURE, wall_top=cfg.FREESLIP, profile=cfg.UNIFORM,
                                               uxInlet_p=0.03, central_moments=cm), ""
    p, g = cfg.womersley_cylinder(central_moments=cm)
    yield "oscillating force with a body", p, g
    # markers half-way between rows: supports whose force is exactly zero
    p, g = cfg.inverted_flag(200, 100, 0.25, 12, Re=100.0, kb=0.6, central_moments=cm)
    yield "flag", p, g


@pytest.mark.parametrize("cm", [0, 1])
def test_single_tiled_step_equals_plain_kernels(gpu_lib, monkeypatch, cm):
    """One step per launch, with support sites, convective outlet and pressure corners."""
    for name, p, g in one_step_cases(cm):
        for prec in (L.LIFE_FP64, L.LIFE_FP32_SHIFTED):
            out = []
            for tile in (None, "0"):
                monkeypatch.delenv("LIFE_TILE", raising=False)
                if tile:
                    monkeypatch.setenv("LIFE_TILE", tile)
                c = Case(p, g, precision=prec)
                c.step(25)
                o = list(c.fields())
                if c.n_markers:
                    m = c.markers()
                    o += [m["pos"], m["force"]]
                c.close()
                out.append(o)
            assert np.isfinite(out[0][0]).all()
            for a, b in zip(*out):
                assert np.array_equal(a, b), (name, cm, prec, float(np.abs(a - b).max()))
