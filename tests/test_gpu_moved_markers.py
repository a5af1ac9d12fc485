"""Markers that the caller moves through the lattice handle of a case, to where
the tiles cannot form the marker forces between the steps of a call (supports in
a convective outlet's column): one call of many steps equals the steps one call
each, bit for bit."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
def test_moved_into_the_outlet_column(gpu_lib, precision):
    p = cfg.lattice_case(96, 60, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.CONVECTIVE, wall_bottom=cfg.WALL,
                         wall_top=cfg.WALL, profile=cfg.UNIFORM, uxInlet_p=0.04, ux0_p=0.03, ref_L=10.0, ref_U=0.04)
    out = []
    for calls in ((1,) * 6, (6,)):
        c = Case(p, "CIRCLE 1 1 40.0 30.0 0.0 0.0 5.0\n", precision=precision)
        c.step(2)
        c.grid.update_markers(c.markers()["pos"] + [50.0, 0.0])
        c.grid.find_support()
        for n in calls:
            c.step(n)
        m = c.markers()
        assert m["supp_ij"][..., 0].max() == c.Nx - 1
        out.append([*c.fields(), m["force"]])
        c.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
