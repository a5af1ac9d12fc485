"""Served cases with one epsilon system over all markers (UNI_EPSILON) and
flexible bodies equal their own life_case run bit for bit, with the FEM on the
device (FP32-shifted populations) and on the host, alone and beside a case whose
bodies have systems of their own."""
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.serve import Server
from tests.test_gpu_serve import assert_same, flag, run_case, served

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
@pytest.mark.parametrize("beside", [False, True])
def test_uniform_epsilon(gpu_lib, precision, beside):
    fsi = cfg.flexible_fsi(Nx=200, Ny=62, D=12.0, centre=(30.0, 30.0), L=42.0, h=2.4, n_el=6, u_mean=0.05, Re=60.0,
                           ramp_steps=0.0, stiffness=2.0, uni_epsilon=1)
    cases = [fsi] + ([flag()] if beside else [])
    ref = [run_case(pg, 15, precision) for pg in cases]
    srv = Server(precision=precision, max_cases=4)
    ids = [srv.submit(p, g, 15, keep_fields=True) for p, g in cases]
    srv.drain()
    for r, rid in zip(ref, ids):
        assert_same(served(srv, rid), r)
    srv.close()
