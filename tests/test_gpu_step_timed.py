"""life_case_step_timed runs the steps of life_case_step: the same state and
step count at the same cost, for lattices that several steps a launch are made
of (both default shapes and the plain kernels), a rigid body, and call lengths
that leave a remainder."""
import time

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case

pytestmark = pytest.mark.gpu


def cavity(N):
    return cfg.lid_driven_cavity(N=N, tau=0.7, u_lid=0.05)


CASES = {"small cavity": (cavity(60), 0), "cavity": (cavity(530), 1),
         "channel": (cfg.cylinder_channel(Nx=200, Ny=64, D=12.0, u_max=0.05, Re=40.0, ramp_steps=0.0, centre=(50.0, 31.5)), 0)}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("every", [0, 7])
def test_same_steps(gpu_lib, name, every):
    (p, g), precision = CASES[name]
    out = []
    for timed in (False, True):
        c = Case(p, g, precision=precision)
        c.set_check_interval(every)
        for n in (1, 23, 4):
            if timed:
                total, kernel = c.step_timed(n)
                assert 0.0 < kernel <= total
            else:
                c.step(n)
        out.append([c.t, *c.fields()])
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("N", [96, 256])
def test_same_cost(gpu_lib, N):
    c = Case(*cavity(N), precision=L.LIFE_FP64)
    n, wall, timed = 1000, [], []
    c.step(n)
    for _ in range(5):
        t0 = time.perf_counter()
        c.step(n)
        wall.append(1e3 * (time.perf_counter() - t0))
        timed.append(c.step_timed(n)[0])
    c.close()
    print("untimed %.2f ms, timed %.2f ms" % (min(wall), min(timed)), flush=True)
    assert min(timed) <= 2.0 * min(wall)  # 3.5 and 2.9 times with a launch per step
