"""Banded epsilon systems whose elimination moves rows, and bands of every width:
exactly the solution of the whole matrix by the host's elimination.  Markers
closer than a spacing, off a line, folded in a zigzag, or with supports cut off
by a wall, placed through a restart file; the number of moved rows and the
half-bandwidth are read off the matrix, so that each case is what it says."""
import struct

import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case

pytestmark = pytest.mark.gpu


def line(n, rng, dx, jx=0.0, jy=0.0, y0=30.0, angle=0.0):
    s = dx * np.arange(n) + jx * rng.uniform(-1, 1, n)
    return np.stack([20.0 + s * np.cos(angle), y0 + s * np.sin(angle) + jy * rng.uniform(-1, 1, n)], axis=1)


def zigzag(n, rng, dx, up, period):
    k = np.arange(n)
    return np.stack([20.0 + dx * k, 30.0 + up * (k % period)], axis=1)


# name: positions, half-bandwidth (most), least part of the rows that move
CASES = {
    "spacing 0.6": (lambda n, r: line(n, r, 0.6, angle=0.5), (5, 5), 0.5),
    "spacing 0.7, off the line": (lambda n, r: line(n, r, 0.7, jy=0.3), (3, 4), 0.3),
    "spacing 0.9, off the line": (lambda n, r: line(n, r, 0.9, 0.2, 0.4), (3, 4), 0.0),
    "spacing 1.3 at a wall": (lambda n, r: line(n, r, 1.3, 0.1, 0.5, y0=-0.5), (2, 2), 0.0),
    "at a wall": (lambda n, r: line(n, r, 0.9, 0.0, 0.3, y0=-0.4), (3, 3), 0.2),
    "zigzag": (lambda n, r: zigzag(n, r, 0.55, 1.0, 2), (5, 5), 0.0),
    "wide zigzag": (lambda n, r: zigzag(n, r, 0.4, 1.3, 3), (6, 8), 0.0),
}


def moved_rows(A):
    """Row exchanges of the elimination with the first largest pivot."""
    A, moved = A.copy(), 0
    for k in range(len(A)):
        p = k + int(np.argmax(np.abs(A[k:, k])))
        assert A[p, k] != 0.0
        if p != k:
            moved += 1
            A[[k, p]] = A[[p, k]]
        rows = k + 1 + np.nonzero(A[k + 1:, k])[0]
        A[rows, k:] -= np.outer(A[rows, k] / A[k, k], A[k, k:])
    return moved


@pytest.mark.parametrize("n", [9, 33, 64, 97, 330])
@pytest.mark.parametrize("name", sorted(CASES))
def test_moved_rows(gpu_lib, tmp_path, name, n):
    make, bw, part = CASES[name]
    pos = make(n, np.random.default_rng(n))
    p = cfg.lattice_case(480, 260, 0.8, wall_left=cfg.VELOCITY, wall_right=cfg.PRESSURE, wall_bottom=cfg.WALL,
                         wall_top=cfg.WALL, profile=cfg.UNIFORM, uxInlet_p=0.01, uni_epsilon=0, ref_L=10.0, ref_U=0.01)
    g = "FILAMENT 1 0 20.0 30.0 0.0 0.0 %.17g 1.0 0.0 FLEXIBLE 4 CLAMPED 10.0 1.0\n" % (n - 1 + 0.5)
    for precision in (L.LIFE_FP64, L.LIFE_FP32_SHIFTED):
        c = Case(p, g, precision=precision)
        assert c.n_markers == n
        c.step(1)
        c.write_restart(str(tmp_path))
        f = tmp_path / "Restart" / "IBM.restart"
        raw = f.read_bytes()
        head = struct.calcsize("=QiQ")
        v = np.frombuffer(raw[head:], dtype=np.float64).reshape(n, 6).copy()
        v[:, :2] = pos
        f.write_bytes(raw[:head] + v.tobytes())
        c.read_restart(str(tmp_path))  # finds the supports and solves for epsilon again
        eps = c.markers()["eps"]
        A = c.grid.epsilon_matrix(0, n)
        c.close()
        r, q = np.nonzero(A)
        width, moved = int(np.abs(r - q).max()), moved_rows(A)
        print(name, n, "half-bandwidth", width, "moved rows", moved, flush=True)
        assert bw[0] <= width <= bw[1] and moved >= part * n
        if precision == L.LIFE_FP32_SHIFTED and width <= 4:
            continue  # cyclic reduction: equal to rounding (test_gpu_eps_cr.py)
        assert np.isfinite(eps).all()
        assert np.array_equal(eps, L.solve_lapack(A, np.ones(n)))
