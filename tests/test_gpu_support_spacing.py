"""Support sites and marker spacing against the oracle, bit for bit: bodies of
one marker, of less and more than a half wavefront's lanes and of more than one
round of positions, markers half-way between sites and supports cut off by the
walls; several bodies, so that workgroups span two."""
import numpy as np
import pytest

from life_amd import config as cfg

pytestmark = pytest.mark.gpu

BODIES = {
    "one marker": [(40.0, 31.5, 0.1)],
    "small": [(40.25, 31.5, 1.1), (70.0, 20.0, 2.3)],
    "around 32": [(40.0, 31.0, 5.0), (70.5, 31.5, 5.3)],
    "two rounds": [(60.0, 31.5, 24.0)],
    "walls": [(20.0, 2.0, 4.0), (100.0, 61.5, 3.0)],
}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(BODIES))
def test_matches_oracle(oracle, gpu_lib, name, precision):
    from life_amd.case import Case
    p, _ = cfg.cylinder_channel(Nx=120, Ny=64, D=16.0, u_max=0.05, Re=40.0, ramp_steps=0.0)
    geom = "".join("CIRCLE 1 %d %.17g %.17g 0.0 0.0 %.17g\n" % (k + 1, *x) for k, x in enumerate(BODIES[name]))
    oc, gc = oracle.OracleCase(p, geom), Case(p, geom, precision=precision)
    m, (cnt, ij, delta) = gc.markers(), oc.supports()
    print(name, "markers", len(cnt), "supports", sorted(set(cnt.tolist())), flush=True)
    assert np.array_equal(m["supp_count"], cnt)
    for k, n in enumerate(cnt):
        assert np.array_equal(m["supp_ij"][k, :n], ij[k, :n]) and np.array_equal(m["supp_delta"][k, :n], delta[k, :n])
    assert np.array_equal(m["ds"], oc.markers()["ds"])
