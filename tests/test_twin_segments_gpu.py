"""The segmented sequential line sweeps (k_twin_seg) against the oracle's
sequential ones: equal values for every line length class (one segment, rows
all in the table, rows that repeat, two lines and one line a workgroup, lines
left to the one-thread-a-line kernel), both axes, 3-D, and data whose warm-up
cannot reach the neighbour's state (exact zeros next to a step), is not
finite or is too small for the quick quotients, where a workgroup sweeps its
lines end to end instead.  Equality is exact (the sign of a zero excepted,
which == does not see).  Which way was taken is checked with the handle's
counts: segments that agree at once for ordinary data, and the three passes
where they are faster."""
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
    if kind == "small":
        return 1e-265 * rng.standard_normal(shp)
    f = np.where(i[0] + i[1] < 0.7, 1.0, -1.0) + 0 * i[2]  # flat on both sides of a step
    if kind == "inf":
        f = f.copy()
        f[shp[0] // 2, shp[1] // 2] = np.inf
    return f


def _check(oracle, ls, ndim, n, h, vel, f, upwind):
    got = ls.compact_derivatives(f, upwind)
    want = [np.zeros(f.size) for _ in range(6)]
    oracle.lib.orc_compact_derivatives(ndim, *n, *h, f.ravel(), *[a.ctypes.data for a in vel], int(upwind), *want)
    for a in range(ndim):
        np.testing.assert_array_equal(got[a].ravel(), want[a])
        np.testing.assert_array_equal(got[3 + a].ravel(), want[3 + a])


def _handle(n):
    ndim = 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 1.3 / n[1], 0.7 / n[2])
    shp = padded_shape(ndim, *n)
    rng = np.random.default_rng(n[0] + n[1])
    vel = [rng.standard_normal(shp) for _ in range(3)]
    ls = LevelSet(ndim, *n, *h)
    ls.set_velocity(*vel)
    return ls, ndim, h, shp, rng, vel


@pytest.mark.parametrize("kind", ["random", "smooth", "step", "inf", "small"])
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_segmented_sweeps_equal_sequential(oracle, n, kind):
    ls, ndim, h, shp, rng, vel = _handle(n)
    f = np.ascontiguousarray(_field(kind, shp, rng), np.float64)
    print(f"segmented sweeps {n} {kind}", flush=True)
    for upwind in (True, False):
        before = ls.line_sweeps()
        _check(oracle, ls, ndim, n, h, vel, f, upwind)
        seg, whole = (b - a for a, b in zip(before, ls.line_sweeps()))
        if max(shp) > (4416 if upwind else 6336):  # lines that do not fit LDS
            assert seg == 0
            continue
        assert seg > 0
        if kind in ("random", "smooth"):
            assert whole == 0
        elif kind != "step" or max(n) > 1000:  # (on short lines every warm-up reaches the ends)
            assert whole > 0


def test_three_passes_where_they_are_faster(oracle):
    """3-D grids of many short lines: one thread a line"""
    n = (48, 40, 52)
    ls, ndim, h, shp, rng, vel = _handle(n)
    print(f"three passes {n}", flush=True)
    for upwind in (True, False):
        _check(oracle, ls, ndim, n, h, vel, rng.standard_normal(shp), upwind)
    assert ls.line_sweeps() == (0, 0)


def test_failed_call_passes_on(oracle):
    """Many long lines: a call in which a workgroup's segments fail is redone
    by the three passes, and the next call starts anew."""
    n = (1400, 1000, 1)
    ls, ndim, h, shp, rng, vel = _handle(n)
    for kind in ("step", "random", "step", "smooth"):
        f = np.ascontiguousarray(_field(kind, shp, rng), np.float64)
        print(f"passed on {n} {kind}", flush=True)
        for upwind in (True, False):
            before = ls.line_sweeps()
            _check(oracle, ls, ndim, n, h, vel, f, upwind)
            seg, whole = (b - a for a, b in zip(before, ls.line_sweeps()))
            assert seg > 0 and (whole > 0) == (kind == "step")


@pytest.mark.parametrize("solver", ["sequential", "partitioned"])
def test_handles_of_different_lengths_in_turn(oracle, solver):
    """the kernels' LDS allowance belongs to the function: a handle of shorter
    lines must not lower it for one of longer lines"""
    shapes = [(1024, 10, 1), (600, 10, 1)]
    hs = [_handle(n) for n in shapes]
    want = [None, None]
    for ls, *_ in hs:
        ls.set_line_solver(solver)
    for turn in range(2):
        for q, (ls, ndim, h, shp, _, vel) in enumerate(hs):
            f = np.ascontiguousarray(_field("random", shp, np.random.default_rng(q)))
            print(f"in turn {shapes[q]} {solver}", flush=True)
            if solver == "sequential":
                for upwind in (True, False):
                    _check(oracle, ls, ndim, shapes[q], h, vel, f, upwind)
                continue
            got = ls.compact_derivatives(f, True)[0]
            assert want[q] is None or np.array_equal(got, want[q])
            want[q] = got
