"""Calls that need an array refuse its absence with an error, as they do any
other bad argument, and accept it where there is nothing to transfer."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case, Grid

pytestmark = pytest.mark.gpu


def test_missing_arrays(gpu_lib):
    lib = L.load()
    p, geom = cfg.cylinder_channel(Nx=120, Ny=64, D=16.0, centre=(40.0, 31.5), u_max=0.05, Re=40.0, ramp_steps=0.0)
    c = Case(p, geom)
    n, eps = c.n_markers, c.markers()["eps"]
    assert lib.life_ibm_set_epsilon(c.grid.h, None) != 0
    assert lib.life_ibm_epsilon_matrix(c.grid.h, 0, n, None) != 0
    assert lib.life_ibm_epsilon_matrix(c.grid.h, 0, 0, None) == 0
    assert lib.life_ibm_update_markers(c.grid.h, None, None) == 0
    assert np.array_equal(c.markers()["eps"], eps)
    c.close()
    g = Grid(p)  # no markers
    assert lib.life_ibm_set_epsilon(g.h, None) == 0
    g.close()
