"""Lattices that the tiles step give what the plain kernels give, bit for bit,
also where the caller has set state by hand: a force outside the supports (an
upload, new markers), which the step after the first leaves out."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Grid

pytestmark = pytest.mark.gpu


def channel(Nx=96, Ny=60, right=cfg.CONVECTIVE):
    return cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.VELOCITY, wall_right=right, wall_bottom=cfg.WALL,
                            wall_top=cfg.WALL, profile=cfg.UNIFORM, uxInlet_p=0.04, ux0_p=0.03, ref_L=10.0, ref_U=0.04)


def ring(x, y, r, n):
    a = 2.0 * np.pi * np.arange(n) / n
    return np.stack([x + r * np.cos(a), y + r * np.sin(a)], axis=1)


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
@pytest.mark.parametrize("how", ["upload", "new markers"])
def test_force_outside_the_supports(gpu_lib, monkeypatch, precision, how):
    p = channel(right=cfg.PRESSURE)
    pos = ring(40.2, 30.1, 6.0, 37)
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    rng = np.random.default_rng(3)
    f = w * (1.0 + 0.01 * rng.standard_normal((p.Nx, p.Ny, 9)))
    u = 0.01 * rng.standard_normal((p.Nx, p.Ny, 2))
    force = 1e-3 * rng.standard_normal((p.Nx, p.Ny, 2))
    out = []
    for tile in (None, "0"):
        monkeypatch.delenv("LIFE_TILE", raising=False)
        if tile:
            monkeypatch.setenv("LIFE_TILE", tile)
        g = Grid(p, precision=precision)
        g.set_markers(pos, np.zeros_like(pos), np.zeros(len(pos)), [1])
        g.find_support()
        g.set_epsilon(np.ones(len(pos)))
        g.upload(f, f.sum(-1), u, force)
        g.lbm_kernel(1)
        if how == "new markers":
            g.interpolate()
            g.spread()
            g.set_markers(pos + 9.0, np.zeros_like(pos), np.zeros(len(pos)), [1])
            g.find_support()
        states = []
        for t in (2, 3):
            g.lbm_kernel(t)
            states += g.download()
        g.set_epsilon(np.ones(len(pos)))
        g.interpolate()
        g.spread()
        g.lbm_kernel(4)
        states += g.download()
        g.close()
        out.append(states)
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
