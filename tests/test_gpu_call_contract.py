"""What the transfer and timing calls promise beside the numbers: a call that
asks for no array still waits for the device, a missing array is an error, and
the timed steps are the steps that life_case_step runs."""
import time

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case, Grid

pytestmark = pytest.mark.gpu


def test_download_of_nothing_waits(gpu_lib):
    lib = L.load()
    g = Grid(cfg.lid_driven_cavity(N=4096, tau=0.7, u_lid=0.05)[0])
    g.sync()
    for call in (lambda: lib.life_grid_download(g.h, None, None, None, None),
                 lambda: lib.life_ibm_download(g.h, *[None] * 8)):
        for t in range(1, 101):  # some 50 ms of work
            g.lbm_kernel(t)
        L.check(call())
        t0 = time.perf_counter()
        g.sync()
        assert time.perf_counter() - t0 < 5e-3
    g.close()


def test_missing_arrays_are_refused(gpu_lib):
    lib = L.load()
    p, geom = cfg.cylinder_channel(Nx=120, Ny=64, D=16.0, centre=(40.0, 31.5), u_max=0.05, Re=40.0, ramp_steps=0.0)
    c = Case(p, geom)
    n, eps = c.n_markers, c.markers()["eps"]
    assert lib.life_ibm_set_epsilon(c.grid.h, None) != 0
    assert np.array_equal(c.markers()["eps"], eps)
    assert lib.life_ibm_epsilon_matrix(c.grid.h, 0, n, None) != 0
    assert lib.life_ibm_epsilon_matrix(c.grid.h, 0, 0, None) == 0
    c.close()
    g = Grid(p)  # no markers: nothing is missing
    assert lib.life_ibm_set_epsilon(g.h, None) == 0
    g.close()


@pytest.mark.parametrize("N", [96, 256])
def test_timed_steps_are_the_untimed_ones(gpu_lib, N):
    c = Case(cfg.lid_driven_cavity(N=N, tau=0.7, u_lid=0.05)[0], "")
    n, wall, timed = 1000, [], []
    c.step(n)
    for _ in range(5):
        t0 = time.perf_counter()
        c.step(n)
        wall.append(1e3 * (time.perf_counter() - t0))
        total, kernel = c.step_timed(n)
        assert 0.0 < kernel <= total
        timed.append(total)
    print("untimed", min(wall), "timed", min(timed), "ms", flush=True)
    assert min(timed) <= 1.4 * min(wall)
    c.close()
    a, b = (Case(cfg.lid_driven_cavity(N=N, tau=0.7, u_lid=0.05)[0], "") for _ in range(2))
    a.set_check_interval(7)
    b.set_check_interval(7)
    a.step(23)
    b.step_timed(23)
    for x, y in zip(a.fields(), b.fields()):
        assert np.array_equal(x, y)
    assert a.t == b.t == 23
    a.close()
    b.close()
