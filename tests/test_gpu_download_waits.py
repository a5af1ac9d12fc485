"""A download that asks for no array still waits for the device: some 50 ms of
queued steps are done when it returns."""
import time

import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("markers", [False, True])
def test_download_of_nothing_waits(gpu_lib, markers):
    lib = L.load()
    g = Grid(cfg.lid_driven_cavity(N=4096, tau=0.7, u_lid=0.05)[0])
    g.sync()
    for t in range(1, 101):
        g.lbm_kernel(t)
    t0 = time.perf_counter()
    if markers:
        L.check(lib.life_ibm_download(g.h, *[None] * 8))
    else:
        L.check(lib.life_grid_download(g.h, None, None, None, None))
    t1 = time.perf_counter()
    g.sync()
    t2 = time.perf_counter()
    print("download %.1f ms, then sync %.1f ms" % (1e3 * (t1 - t0), 1e3 * (t2 - t1)), flush=True)
    assert t2 - t1 < 5e-3
    g.close()
