"""Banded epsilon systems on the device (plain method): exactly the solution of
the whole matrix by the host's elimination, for filaments of fewer rows than
the window, around the half and whole wavefront, and past the rows that fit in
LDS, at angles that give half-bandwidths 2 and 3."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [2, 4, 31, 32, 33, 62, 63, 64, 96, 97, 130, 290, 330])
@pytest.mark.parametrize("angle,bw", [(180, 2), (150, 3), (135, 3)])
def test_matches_whole_matrix(gpu_lib, tmp_path, length, angle, bw):
    from life_amd.case import Case
    Ny = 2 * length + 24
    p, g = cfg.inverted_flag(Nx=int(2.5 * length) + 40, Ny=Ny, length_frac=(length + 0.5) / Ny, n_el=max(2, length // 8),
                             Re=100.0, kb=0.3)
    g = g.replace(" 180.0 FLEXIBLE", " %.1f FLEXIBLE" % angle)
    c = Case(p, g)
    c.step(3)
    c.write_restart(str(tmp_path))
    d = Case(p, g)
    d.read_restart(str(tmp_path))  # finds the supports and solves for epsilon again
    n, eps = d.n_markers, d.markers()["eps"]
    d.grid.n_markers = n
    A = d.grid.epsilon_matrix(0, n)
    r, q = np.nonzero(A)
    print("markers", n, "half-bandwidth", int(np.abs(r - q).max()), flush=True)
    assert n == length + 1 and np.abs(r - q).max() <= bw
    assert np.array_equal(eps, lib.solve_lapack(A, np.ones(n)))
