"""State and marker transfers (chunks of sites through page-locked buffers):
lattices of one chunk, of exactly and just past a chunk's sites, and of more
chunks than buffers; each output alone and all together; an upload followed by
a download gives the same numbers back."""
import ctypes as C

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case, Grid

pytestmark = pytest.mark.gpu


# one 64 KiB chunk; 16 MiB chunks hold 149 760 sites of a whole state (14 doubles each) and 699 008 of rho and u
@pytest.mark.parametrize("Nx,Ny", [(4, 4), (37, 15), (585, 256), (150, 999), (1030, 1021)])
def test_upload_download_round_trip(gpu_lib, Nx, Ny):
    p = cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE, wall_bottom=cfg.WALL,
                         wall_top=cfg.FREESLIP, profile=cfg.UNIFORM, uxInlet_p=0.03)
    rng = np.random.default_rng(Nx)
    f = rng.uniform(0.01, 0.4, (Nx, Ny, 9))
    rho, u, b = f.sum(-1), rng.standard_normal((Nx, Ny, 2)), rng.standard_normal((Nx, Ny, 2))
    g = Grid(p)
    g.upload(f, rho, u, b)
    for a, e in zip(g.download(), (f, rho, u, b)):
        assert np.array_equal(a, e)
    lib, dp = L.load(), L.dptr
    for k in range(4):  # one output at a time
        out = [np.zeros_like(x) for x in (f, rho, u, b)]
        args = [dp(out[q]) if q == k else None for q in range(4)]
        L.check(lib.life_grid_download(g.h, *args))
        assert np.array_equal(out[k], (f, rho, u, b)[k])
    L.check(lib.life_grid_download(g.h, None, None, None, None))
    g.upload(f, rho, u)  # no force: zero
    assert not g.download()[3].any()
    g.close()


def test_fp32_state_keeps_the_shift(gpu_lib):
    p = cfg.lattice_case(61, 47, 0.7, wall_left=cfg.FLUID, wall_right=cfg.FLUID, wall_bottom=cfg.FLUID,
                         wall_top=cfg.FLUID, profile=cfg.UNIFORM, uxInlet_p=0.0)
    rng = np.random.default_rng(5)
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    f = w * (1.0 + 0.05 * rng.standard_normal((61, 47, 9)))
    g = Grid(p, precision=L.LIFE_FP32_SHIFTED)
    g.upload(f, f.sum(-1), np.zeros((61, 47, 2)))
    assert np.array_equal(g.download()[0], (f - w).astype(np.float32).astype(np.float64) + w)
    g.close()


def test_marker_arrays(gpu_lib):
    p, geom = cfg.cylinder_channel(Nx=120, Ny=64, D=16.0, centre=(40.0, 31.5), u_max=0.05, Re=40.0, ramp_steps=0.0)
    c = Case(p, geom)
    c.step(3)
    m = c.markers()
    n = c.n_markers
    g = c.grid
    only = np.zeros((n, 2))
    L.check(L.load().life_ibm_download(g.h, None, None, L.dptr(only), None, None, None, None, None))
    assert np.array_equal(only, m["force"]) and np.abs(only).max() > 0
    pos, vel = m["pos"] + 0.25, m["vel"] + 0.5
    for k in range(3):  # queued one after the other: the last one stands
        g.update_markers(pos - 1.0 + 0.5 * k, None)
    g.update_markers(None, vel)
    again = g.markers(n)
    assert np.array_equal(again["pos"], pos) and np.array_equal(again["vel"], vel)
    g.set_epsilon(np.arange(n) * 0.5)
    assert np.array_equal(g.markers(n)["eps"], np.arange(n) * 0.5)
    c.close()
