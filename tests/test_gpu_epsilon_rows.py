"""Epsilon systems solved from their non-zeros: exactly the solution of the
whole matrix, for systems around a wavefront of columns, of sizes that leave
rows over in a workgroup, one body or several in a system, and with many
non-zeros a row (circles a quarter of a spacing apart)."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uni,circles", [
    (0, [(60.0, 31.5, 1.6)]), (0, [(60.0, 31.5, 10.1)]), (0, [(60.0, 31.5, 10.2), (90.3, 31.5, 10.35)]),
    (1, [(40.0, 31.5, 8.0), (80.2, 30.9, 12.7)]),
    (1, [(60.0, 31.5, 9.0 + 0.25 * k) for k in range(6)]),
])
def test_rows_give_the_dense_solution(gpu_lib, uni, circles):
    from life_amd.case import Case
    p, _ = cfg.cylinder_channel(Nx=120, Ny=64, D=16.0, u_max=0.05, Re=40.0, ramp_steps=0.0)
    geom = "".join("CIRCLE 1 %d %.17g %.17g 0.0 0.0 %.17g\n" % (k + 1, *c) for k, c in enumerate(circles))
    c = Case(p.replace(uni_epsilon=uni), geom)
    n, eps = c.n_markers, c.markers()["eps"]
    c.grid.n_markers = n
    if uni:
        systems = [(0, n)]
    else:
        systems = [(c.body_info(b)["first"], c.body_info(b)["n"]) for b in range(c.n_bodies)]
    for first, m in systems:
        A = c.grid.epsilon_matrix(first, m)
        print("system", m, "most non-zeros in a row", int((A != 0).sum(1).max()), flush=True)
        assert np.array_equal(eps[first:first + m], lib.solve_lapack(A, np.ones(m)))
