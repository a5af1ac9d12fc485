"""A served case whose FEM runs on the device goes on from its present state when
a case is admitted whose beam does not fit the device FEM (all of them take the
host's FEM then), and back on the device when that case has left: the trajectory
is that of its own life_case run.  Bar 1e-9 relative, that of
test_gpu_fem_device.py: the two FEMs agree to the rounding of their solves."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.serve import Server
from tests._util import rel_err
from tests.test_gpu_serve import flag, run_case, served

pytestmark = pytest.mark.gpu

BAR = 1e-9


def long_beam():
    """One beam of 200 elements: more than the device FEM's LDS holds."""
    p, g = cfg.canopy(Nx=160, Ny=420, n_filaments=1, L=400.0, n_el=200, min_spacing=30.0, x_range=(60, 100),
                      ramp_steps=0.0, u_in=0.02, kb_range=(5e-2, 5e-2))
    return p.replace(ux0_p=0.02), g


def test_switch_and_back(gpu_lib):
    x, steps = flag(Nx=192, Ny=96, n_el=10, Re=200.0, kb=0.3), 30
    ref = run_case(x, steps, L.LIFE_FP32_SHIFTED)
    srv = Server(precision=L.LIFE_FP32_SHIFTED, max_cases=4)
    rid = srv.submit(*x, steps, keep_fields=True)
    for _ in range(8):
        srv.step()
    other = srv.submit(*long_beam(), 9)
    srv.drain()
    assert srv.info(other)["status"] == L.LIFE_REQ_DONE, srv.error(other)
    got = served(srv, rid)
    srv.close()
    errs = {k: rel_err(got[k], ref[k]) for k in ref}
    print(errs, flush=True)
    assert np.abs(ref["pos"] - run_case(x, 1, L.LIFE_FP32_SHIFTED)["pos"]).max() > 1e-3
    assert max(errs.values()) <= BAR, errs
