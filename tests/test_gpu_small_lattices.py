"""Lattices at the edges of the boundary kernel's split (seven sites per
wavefront, nine lanes each): site counts that fill the last wavefront, leave
one site in it or none, and sides so short that corners share neighbours.
Every boundary type, both operators, FP64 against the oracle at the parity
bar (1e-12 relative: same operations in the same order)."""
import numpy as np
import pytest

from life_amd import lib as L
from life_amd.case import Case
from tests._util import BC_KINDS, bc_mix_params, rel_err

pytestmark = pytest.mark.gpu

# boundary sites 2 (Nx + Ny) - 4: 14 = 2 x 7, 16, 22 = 3 x 7 + 1, 27 x 7 = 189 + 1 ...
SIZES = [(5, 4), (6, 4), (8, 5), (70, 27)]


@pytest.mark.parametrize("cm", [0, 1])
@pytest.mark.parametrize("kind", BC_KINDS)
def test_boundary_sites_of_small_lattices(oracle, gpu_lib, kind, cm):
    for Nx, Ny in SIZES:
        p, g = bc_mix_params(kind, Nx=Nx, Ny=Ny, cm=cm)
        steps = 25
        oc = oracle.OracleCase(p, g)
        oc.step(steps)
        gc = Case(p, g, precision=L.LIFE_FP64)
        gc.step(1)
        gc.step(steps - 1)
        f, rho, u, _ = gc.fields()
        fo, ro, uo, _ = oc.grid()
        assert np.isfinite(f).all()
        for a, b in ((f, fo), (rho, ro), (u, uo)):
            assert rel_err(a, b) <= 1e-12, (kind, cm, Nx, Ny)
        gc.close()
        oc.close()
