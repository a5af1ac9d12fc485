"""Lattices and served batches of so many boundary sites that the boundary
kernel takes one lane per site: bit for bit the nine lanes' values, which the
tiles form with the same arithmetic, for every boundary type, first steps on an
uploaded state, and lattices just below and above the line (24 000 sites in FP64,
36 000 in FP32)."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case
from life_amd.serve import Server
from tests._util import BC_KINDS, bc_mix_params

pytestmark = pytest.mark.gpu


def params(kind, Nx, Ny, cm):
    if kind == "pressure_corners":
        return cfg.lattice_case(Nx, Ny, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE, wall_bottom=cfg.PRESSURE,
                                wall_top=cfg.FREESLIP, profile=cfg.UNIFORM, uxInlet_p=0.03, central_moments=cm)
    return bc_mix_params(kind, Nx=Nx, Ny=Ny, cm=cm)[0]


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
@pytest.mark.parametrize("cm", [0, 1])
@pytest.mark.parametrize("kind", BC_KINDS + ["pressure_corners"])
def test_equals_the_tiles(gpu_lib, monkeypatch, kind, cm, precision):
    line = 24000 if precision == L.LIFE_FP64 else 36000
    for n in (line - 2, line + 10, 3 * line):
        p = params(kind, n // 2, 6, cm)
        rng = np.random.default_rng(n)
        w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
        f = w * (1.0 + 0.02 * rng.standard_normal((p.Nx, p.Ny, 9)))
        state = (f, f.sum(-1), 0.01 * rng.standard_normal((p.Nx, p.Ny, 2)))
        out = []
        for tile in (False, True):
            if tile:
                monkeypatch.delenv("LIFE_TILE")
                monkeypatch.setenv("LIFE_TILE1", "14,30")
            else:
                monkeypatch.delenv("LIFE_TILE1", raising=False)
                monkeypatch.setenv("LIFE_TILE", "0")
            c = Case(p, "", precision=precision)
            c.grid.upload(*state)
            for t in range(1, 6):
                c.grid.lbm_kernel(t)
            out.append(c.fields())
            c.close()
        assert np.isfinite(out[0][0]).all()
        for a, b in zip(*out):
            assert np.array_equal(a, b), (n, float(np.abs(a - b).max()))


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
def test_served_batch(gpu_lib, precision):
    """80 cases of some 1100 boundary sites, 40 of each collision operator: each as it is alone."""
    cases = [params(k, 520, 37 + q % 3, cm) for q in range(10) for k in ("channel_convective", "channel_pressure",
                                                                         "shear_velocity", "pressure_corners")
             for cm in (0, 1)]
    srv = Server(precision=precision, max_cases=len(cases))
    ids = [srv.submit(p, "", 6, keep_fields=True) for p in cases]
    srv.drain()
    assert srv.stats()["peak_running"] == len(cases)
    for p, rid in list(zip(cases, ids))[::3]:
        c = Case(p, "", precision=precision)
        c.step(6)
        _, rho, u, _ = c.fields()
        c.close()
        srho, su, _ = srv.fields(rid)
        assert np.array_equal(srho, rho) and np.array_equal(su, u)
    srv.close()
