"""Rigid bodies that overlap, touch, lie within each other or at the walls, up to
just under the crowd at which the tiles leave the marker forces to launches of
their own (128 markers around a tile): a call of five steps equals five calls, and
the spread of the last step equals the sums in marker order, bit for bit, while
every value is finite."""
import numpy as np
import pytest

from life_amd import config as cfg
from life_amd import lib as L
from life_amd.case import Case

pytestmark = pytest.mark.gpu

STEPS = 5
CASES = {
    "overlapping": [(40.0 + 1.3 * k, 30.0 + 0.7 * k, 5.0 + 1.1 * k) for k in range(3)],
    "touching": [(30.0, 30.0, 6.0), (42.6, 30.2, 6.0), (36.3, 19.2, 6.0)],
    "at the walls": [(20.0, 5.0, 4.0), (70.0, 57.9, 5.0)],
    "nested": [(40.0, 31.5, 2.0 + 1.5 * k) for k in range(4)],
    "nested wide": [(40.0, 31.5, 2.0 + 2.0 * k) for k in range(4)],
    "crowd": [(30 + 9.3 * (k % 3), 20 + 9.3 * (k // 3), 3.2) for k in range(6)],
}


def around_a_tile(pos):
    """Most markers in two by two buckets of 20 x 36 sites (forces_suit_tiles)."""
    b, n = np.unique(np.stack([pos[:, 0] // 20, pos[:, 1] // 36], axis=1).astype(int), axis=0, return_counts=True)
    count = dict(zip(map(tuple, b), n))
    return max(sum(count.get((i + p, j + q), 0) for p in (0, 1) for q in (0, 1)) for i in range(-1, 7) for j in range(-1, 3))


def in_marker_order(c):
    m = c.markers()
    out = np.zeros_like(c.fields()[3])
    k, s = np.nonzero(np.arange(9)[None, :] < m["supp_count"][:, None])
    i, j = m["supp_ij"][k, s].T
    for x in range(2):
        np.add.at(out[..., x], (i, j), m["force"][k, x] * m["eps"][k] * m["ds"][k] * 1.0 * m["supp_delta"][k, s])
    return out


@pytest.mark.parametrize("precision", [L.LIFE_FP64, L.LIFE_FP32_SHIFTED])
@pytest.mark.parametrize("right", [cfg.CONVECTIVE, cfg.PRESSURE])
@pytest.mark.parametrize("name", sorted(CASES))
def test_call_of_many_steps(gpu_lib, name, right, precision):
    p = cfg.lattice_case(120, 64, 0.7, wall_left=cfg.VELOCITY, wall_right=right, wall_bottom=cfg.WALL,
                         wall_top=cfg.WALL, profile=cfg.UNIFORM, uxInlet_p=0.02, ux0_p=0.02, central_moments=1,
                         ref_L=10.0, ref_U=0.04)
    geom = "".join("CIRCLE 1 %d %.17g %.17g 0.0 0.0 %.17g\n" % (k + 1, *x) for k, x in enumerate(CASES[name]))
    out = []
    for calls in ((1,) * STEPS, (STEPS,), (2, 3)):
        c = Case(p, geom, precision=precision)
        for n in calls:
            c.step(n)
        m = c.markers()
        assert c.n_markers <= 256 and around_a_tile(m["pos"]) <= 128
        if name == "at the walls":
            assert {0, 63} & set(m["supp_ij"][..., 1][np.arange(9)[None, :] < m["supp_count"][:, None]])
        state = [*c.fields(), m["force"], m["eps"], c.total_force()]
        assert all(np.isfinite(x).all() for x in state) and np.abs(m["force"]).max() > 0.0
        assert np.array_equal(state[3], in_marker_order(c))
        out.append(state)
        c.close()
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)
