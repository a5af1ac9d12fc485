"""Rigid bodies stepped many steps in a call (the tiles form the marker forces
between the steps) against the same steps one call each (interpolation and
spread of their own), bit for bit (bodies cut by a
wall or laid over each other end in NaN, at the same sites): both storages and collision operators, few
and many markers, bodies at walls, across tiles and at the edges of a periodic
lattice, near a convective outlet, too many markers, a force left over from an
upload, a body force."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd.case import Case

pytestmark = pytest.mark.gpu


def lattice(Nx, Ny, right=cfg.CONVECTIVE, cm=1, **kw):
    periodic = right == cfg.FLUID
    side = dict(wall_left=cfg.FLUID, wall_right=cfg.FLUID, wall_bottom=cfg.FLUID, wall_top=cfg.FLUID) if periodic else dict(
        wall_left=cfg.VELOCITY, wall_right=right, wall_bottom=cfg.WALL, wall_top=cfg.WALL)
    return cfg.lattice_case(Nx, Ny, 0.7, profile=cfg.UNIFORM, uxInlet_p=0.04, ux0_p=0.03, central_moments=cm, ref_L=10.0,
                            ref_U=0.04, **side).replace(**kw)


def circles(*c):
    return "".join("CIRCLE 1 %d %.17g %.17g 0.0 0.0 %.17g\n" % (k + 1, *x) for k, x in enumerate(c))


CASES = {
    "one marker pair": (lattice(96, 48), circles((30.0, 23.5, 0.4))),
    "cylinder": (lattice(120, 64), circles((40.3, 31.2, 8.0))),
    "cylinder bgk": (lattice(120, 64, cm=0), circles((40.3, 31.2, 8.0))),
    "pressure outlet": (lattice(120, 64, right=cfg.PRESSURE), circles((40.3, 31.2, 8.0), (70.0, 20.0, 6.5))),
    "at the walls": (lattice(120, 64), circles((20.0, 3.0, 4.0), (70.0, 61.0, 5.0))),
    "at the outlet": (lattice(96, 48), circles((91.0, 23.5, 3.0))),
    "into the outlet": (lattice(96, 48), circles((93.0, 23.5, 3.0))),
    "periodic": (lattice(70, 50, right=cfg.FLUID), circles((3.0, 2.5, 3.0), (66.5, 46.0, 3.5), (30.0, 25.0, 6.0))),
    "dense": (lattice(120, 64), circles(*[(40.0 + 0.9 * k, 30.0 + 0.3 * k, 5.0 + 0.6 * k) for k in range(4)])),
    "piled up": (lattice(120, 64), circles(*[(40.0, 31.5, 1.0 + 0.55 * k) for k in range(11)])),
    "too many": (lattice(240, 128), circles((60.0, 63.5, 30.0), (150.0, 63.5, 31.0))),
    "larger lattice": (lattice(620, 300), circles((100.2, 150.1, 15.0), (180.0, 120.0, 9.0))),
    "body force": (lattice(120, 64, right=cfg.PRESSURE, gravityX=1e-6, gravityY=-2e-6), circles((40.3, 31.2, 8.0))),
}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(CASES))
def test_call_of_many_steps(gpu_lib, name, precision):
    p, geom = CASES[name]
    out = []
    for calls in ((1,) * 12, (12,), (2, 7, 3)):
        c = Case(p, geom, precision=precision)
        for k, n in enumerate(calls):
            c.step(n)
            if len(calls) == 3 and k == 0:
                f, rho, u, b = c.fields()
                c.grid.upload(f, rho, u, b)  # the force comes back as it was
        m = c.markers()
        out.append([*c.fields(), m["force"], m["eps"], c.total_force()])
        print(name, "markers", c.n_markers, flush=True)
        c.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b, equal_nan=True)
    if precision == 0:  # (an upload rounds FP32 deviations)
        for a, b in zip(out[0], out[2]):
            assert np.array_equal(a, b, equal_nan=True)
