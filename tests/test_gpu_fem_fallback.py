"""Epsilon systems that are not banded (a filament folded onto itself) with the
FEM on the device: the host solves the whole system once the device FEM has
reported it, and the FEM runs again with that epsilon.  Supports, positions and
epsilon are those of the coupling's start then, as with the host FEM, so both
give the same step.  Bar 1e-9 relative, that of test_gpu_fem_device.py: the two
FEMs agree to the rounding of their linear solves."""
import struct

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case
from tests._util import rel_err

pytestmark = pytest.mark.gpu

BAR = 1e-9
ROOT = np.array([30.0, 40.0])


def straight():
    """A soft filament of 41 markers on 8 elements along a channel's axis."""
    p = cfg.lattice_case(120, 80, 0.8, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE, wall_bottom=cfg.FREESLIP,
                         wall_top=cfg.FREESLIP, profile=cfg.UNIFORM, uxInlet_p=0.02, uyInlet_p=0.02, ux0_p=0.02,
                         uy0_p=0.02, uni_epsilon=0, ref_L=40.0, ref_U=0.02, subTol=1e-6)
    return p, "FILAMENT 1 0 %.17g %.17g 0.0 0.0 40.0 1.0 0.0 FLEXIBLE 8 CLAMPED 50.0 1e-6\n" % tuple(ROOT)


def fold(path):
    """Lay the filament of the FEM state file back along itself, two spacings above."""
    xy = np.array([(5 * k, 0) for k in range(5)] + [(20, 2)] + [(15 - 5 * k, 2) for k in range(3)], float) + ROOT
    node_a = np.array([0.0] * 4 + [np.pi / 4, 3 * np.pi / 4] + [np.pi] * 3)
    el_a = np.array([0.0] * 4 + [np.pi / 2] + [np.pi] * 3)
    raw = path.read_bytes()
    head = struct.calcsize("=idiQQ")
    _, _, _, nel, nnode = struct.unpack("=idiQQ", raw[:head])
    assert (nel, nnode) == (8, 9)
    v = np.frombuffer(raw[head:], dtype=np.float64).copy()
    U, node = v[:6 * 27].reshape(6, 27), v[-54:].reshape(9, 6)
    move = np.concatenate([xy - node[:, :2], (node_a - node[:, 4])[:, None]], axis=1).ravel()
    for k in (0, 3, 4):  # U, Un, Unm1
        U[k] = move
    el = v[6 * 27:-54].reshape(8, 2)
    el[:, 0] = np.hypot(*np.diff(xy, axis=0).T)
    el[:, 1] = el_a
    node[:, 2:4] = xy
    node[:, 5] = node_a
    path.write_bytes(raw[:head] + v.tobytes())


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
def test_folded_filament(gpu_lib, tmp_path, monkeypatch, precision):
    p, g = straight()
    c = Case(p, g, precision=precision)
    c.step(3)
    c.write_restart(str(tmp_path))
    c.close()
    fold(tmp_path / "Restart" / "FEM.restart")
    out = []
    for device in (0, 1):
        monkeypatch.setenv("LIFE_DEVICE_FEM", str(device))
        c = Case(p, g, precision=precision)
        c.read_restart(str(tmp_path))
        steps = []
        for _ in range(4):
            c.step(1)
            m = c.markers()
            A = c.grid.epsilon_matrix(0, c.n_markers)
            r, q = np.nonzero(A)
            print("device" if device else "host", "half-bandwidth", int(np.abs(r - q).max()), "largest move",
                  float(np.abs(m["vel"]).max()), c.coupling(), flush=True)
            assert np.abs(r - q).max() > 8  # wider than the band
            assert np.isfinite(m["eps"]).all()
            steps.append([m["eps"], m["pos"], m["force"], c.fields()[2]])
        out.append(steps)
        c.close()
    for host, device in zip(*out):
        errs = [rel_err(b, a) for a, b in zip(host, device)]
        print(errs, flush=True)
        assert max(errs) <= BAR
