"""The spread of markers that a caller sets in any order: sums in marker order,
bit for bit, up to and past the number that is compared marker by marker, and no
dearer there than by the passes over lists, which more markers take."""
import time

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Grid

pytestmark = pytest.mark.gpu


def scattered(n, seed=1):
    p = cfg.lattice_case(560, 560, 0.7, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE, wall_bottom=cfg.WALL,
                         wall_top=cfg.WALL, profile=cfg.UNIFORM, uxInlet_p=0.02, ux0_p=0.02, central_moments=1)
    g = Grid(p, precision=L.LIFE_FP64)
    pos = 30.0 + 500.0 * np.random.default_rng(seed).uniform(size=(n, 2))
    g.set_markers(pos, np.zeros_like(pos), np.zeros(n), [1])
    g.find_support()
    g.set_epsilon(np.linspace(1.0, 2.0, n))
    g.lbm_kernel(1)
    return g


@pytest.mark.parametrize("n", [4999, 5000, 5001, 8192])
def test_sums_in_marker_order(gpu_lib, n):
    g = scattered(n)
    g.interpolate()
    g.spread()
    m, got = g.markers(n), g.download()[3]
    want = np.zeros_like(got)
    k, s = np.nonzero(np.arange(9)[None, :] < m["supp_count"][:, None])
    i, j = m["supp_ij"][k, s].T
    for x in range(2):
        np.add.at(want[..., x], (i, j), m["force"][k, x] * m["eps"][k] * m["ds"][k] * 1.0 * m["supp_delta"][k, s])
    assert np.isfinite(got).all() and got.any()
    assert np.array_equal(got, want)
    g.close()


def test_cost(gpu_lib):
    us = {}
    for n in (8192, 9000):
        g = scattered(n)
        best = 1e9
        for _ in range(8):
            t0 = time.perf_counter()
            for _ in range(40):
                g.spread()
            g.sync()
            best = min(best, time.perf_counter() - t0)
        us[n] = best / 40e-6
        g.close()
    print(us, flush=True)
    assert us[8192] <= 1.2 * us[9000]  # 1.45 times when each marker was compared with all
