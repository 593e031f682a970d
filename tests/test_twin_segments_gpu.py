"""The segmented sequential line sweeps (k_twin_seg) against the oracle's
sequential ones: equal values for every line length class (one segment, rows
all in the table, rows that repeat, two lines and one line a workgroup, lines
left to the one-thread-a-line kernel), both axes, 3-D, and data whose warm-up
cannot reach the neighbour's state (exact zeros next to a step) or is not
finite, where a workgroup sweeps sequentially instead.  Equality is exact (the
sign of a zero excepted, which == does not see)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.pyoracle import Oracle
from scihpc_amd import LevelSet, padded_shape

SHAPES = [(12, 9, 1), (90, 91, 1), (91, 300, 1), (1024, 10, 1), (10, 1031, 1), (2100, 7, 1), (7, 4200, 1),
          (5000, 6, 1), (14, 40, 33)]


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


def _field(kind, shp, rng):
    if kind == "random":
        return rng.standard_normal(shp)
    i = [np.arange(m).reshape([-1 if d == e else 1 for e in range(3)]) / max(shp) for d, m in enumerate(shp)]
    if kind == "smooth":
        return np.sin(7 * i[0]) * np.cos(5 * i[1] + i[2]) + 0 * i[2]
    f = np.where(i[0] + i[1] < 0.7, 1.0, -1.0) + 0 * i[2]  # flat on both sides of a step
    if kind == "inf":
        f = f.copy()
        f[shp[0] // 2, shp[1] // 2] = np.inf
    return f


@pytest.mark.parametrize("kind", ["random", "smooth", "step", "inf"])
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_segmented_sweeps_equal_sequential(oracle, n, kind):
    ndim = 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 1.3 / n[1], 0.7 / n[2])
    shp = padded_shape(ndim, *n)
    rng = np.random.default_rng(n[0] + n[1])
    f = np.ascontiguousarray(_field(kind, shp, rng), np.float64)
    vel = [rng.standard_normal(shp) for _ in range(3)]
    print(f"segmented sweeps {n} {kind}", flush=True)
    ls = LevelSet(ndim, *n, *h)
    ls.set_velocity(*vel)
    for upwind in (True, False):
        got = ls.compact_derivatives(f, upwind)
        want = [np.zeros(shp).ravel() for _ in range(6)]
        oracle.lib.orc_compact_derivatives(ndim, *n, *h, f.ravel(), *[a.ctypes.data for a in vel],
                                           int(upwind), *want)
        for a in range(ndim):
            np.testing.assert_array_equal(got[a].ravel(), want[a])
            np.testing.assert_array_equal(got[3 + a].ravel(), want[3 + a])
