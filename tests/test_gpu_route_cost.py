"""The route that a lattice takes by itself is not slower than the plain kernels
(LIFE_TILE=0): long lattices of few sites across, where every tile has a
boundary, and periodic ones, whose plain step is a single launch.  1.25 times the
plain step leaves room for the timer; the tiles took 1.2 to 3.3 times here."""
import time

import pytest

from life_amd import config as cfg
from life_amd.case import Case

pytestmark = pytest.mark.gpu


def cavity(Nx, Ny, cm):
    return cfg.lid_driven_cavity(N=Ny, tau=0.7, u_lid=0.05, central_moments=cm)[0].replace(Nx=Nx)


def periodic(Nx, Ny, cm):
    return cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.FLUID, wall_right=cfg.FLUID, wall_bottom=cfg.FLUID,
                            wall_top=cfg.FLUID, profile=cfg.UNIFORM, uxInlet_p=0.0, ux0_p=0.03, central_moments=cm)


def outlet(Nx, Ny, cm):
    return cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.CONVECTIVE, wall_bottom=cfg.WALL,
                            wall_top=cfg.FREESLIP, profile=cfg.UNIFORM, uxInlet_p=0.05, central_moments=cm)


@pytest.mark.parametrize("make,Nx,Ny,cm,precision", [
    (cavity, 4, 300000, 0, 0), (cavity, 300000, 4, 1, 1), (cavity, 8, 62501, 0, 1), (cavity, 25001, 112, 1, 1),
    (periodic, 50001, 12, 0, 1), (periodic, 1300, 2154, 1, 1), (outlet, 200000, 4, 0, 0), (outlet, 50001, 8, 1, 1),
])
def test_not_slower_than_plain(gpu_lib, monkeypatch, make, Nx, Ny, cm, precision):
    c = Case(make(Nx, Ny, cm), "", precision=precision)
    c.set_check_interval(0)
    best = {}
    for tile in (None, "0") * 5:
        monkeypatch.delenv("LIFE_TILE", raising=False)
        if tile:
            monkeypatch.setenv("LIFE_TILE", tile)
        t0 = time.perf_counter()
        c.step(60)
        best[tile] = min(best.get(tile, 1e9), time.perf_counter() - t0)
    c.close()
    print("own route %.1f us a step, plain %.1f" % (best[None] / 60e-6, best["0"] / 60e-6), flush=True)
    assert best[None] <= 1.25 * best["0"]
