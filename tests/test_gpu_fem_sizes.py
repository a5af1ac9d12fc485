"""The device FEM against the host FEM over numbers of elements at the edges of
its splits: chains of one level of the reduction and of node counts around its
rounds, bodies around the elements of one round of rows with both workgroup
sizes, more load-map entries than fit beside the solve, and many bodies."""
import numpy as np
import pytest

from life_amd import config as cfg
from tests._util import rel_err
from tests.test_gpu_fem_device import BAR, run

pytestmark = pytest.mark.gpu


def flag(length, n_el):
    return cfg.inverted_flag(Nx=3 * length + 40, Ny=2 * length + 24, length_frac=(length + 0.5) / (2 * length + 24),
                             n_el=n_el, Re=100.0, kb=0.5)


def filaments(n, n_el):
    p, g = cfg.canopy(Nx=40 * n + 80, Ny=96, n_filaments=n, L=48.0, n_el=n_el, min_spacing=36.0,
                      x_range=(40, 40 + 38 * n), ramp_steps=0.0, u_in=0.05, kb_range=(1e-1, 3e-1))
    return p.replace(ux0_p=0.05), g


CASES = {"n%d on %d" % (e, m): (lambda m=m, e=e: flag(m, e))
         for m, e in [(24, 1), (24, 2), (24, 3), (60, 2), (60, 12), (60, 13), (60, 27), (60, 41), (60, 42), (60, 43),
                      (100, 84), (100, 85), (100, 86)]}
CASES["32 bodies"] = lambda: filaments(32, 43)
CASES["33 bodies"] = lambda: filaments(33, 43)


@pytest.mark.parametrize("name", sorted(CASES))
def test_device_fem_sizes(monkeypatch, gpu_lib, name):
    pg = CASES[name]()
    h, d = run(pg, 5, monkeypatch, False), run(pg, 5, monkeypatch, True)
    errs = {k: rel_err(d[k], h[k]) for k in ("u", "pos", "force", "U")}
    print(name, d["subits"], " ".join("%s %.2g" % kv for kv in errs.items()), flush=True)
    assert d["subits"] == h["subits"]
    for k, e in errs.items():
        assert e <= BAR, (k, e)
