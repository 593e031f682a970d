"""The fused redistancing stage (k_redist2d) and the in-place one of 1-D and
3-D (k_redist_stage) against the oracle at the edges of the 16 x 32 tiles (14 x
30 cells of the padded range are advanced), on the smallest grids, under
every boundary condition, mixed over the sides, and for level sets whose
smoothness terms leave the range of a double when multiplied (k_godunov's
weights).

Bar: 1e-12 of the largest value after two steps.  A gradient is formed from
about 60 FP64 operations an axis in another order than the oracle's (each
slope to a few ulp of max|phi| / h), and enters the level set times rdt = h /
4 in each of six stages: some 1e-14, with room for the quotient a / b."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.pyoracle import Oracle
from scihpc_amd import LevelSet, padded_shape
from scihpc_amd._capi import BC_CODES

SHAPES = [(3, 3, 1), (8, 24, 1), (9, 25, 1), (22, 54, 1), (23, 55, 1), (37, 84, 1), (40, 1, 1), (5, 9, 7), (12, 10, 33)]
BCS = [["neumann"] * 6, ["periodic"] * 6, ["no_slip", "slip", "neumann", "no_slip", "slip", "neumann"],
       ["dirichlet", "neumann", "slip", "dirichlet", "neumann", "dirichlet"]]


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


def _run(oracle, n, bc, scale, steps):
    ndim = 1 if n[1] == 1 else 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 0.8 / n[1], 1.1 / n[2])
    shp = padded_shape(ndim, *n)
    x = np.indices(shp)
    r2 = sum(((x[a] - 2.5) * h[a] - 0.4) ** 2 for a in range(ndim))
    phi = scale * (0.3 - np.sqrt(r2)) * (1.0 + 0.2 * np.sin(3.0 * x[0] * h[0]))
    width, dt, rdt = 1.5 * h[0], 0.1 * h[0], 0.25 * h[0]
    vals = np.linspace(-0.3, 0.4, 6)
    types = np.array([BC_CODES[b] for b in bc], np.int32)
    print(f"redistance {n} {bc} {scale:g}", flush=True)
    ls = LevelSet(ndim, *n, *h, bc, list(vals))
    ls.set_phi(phi)
    want = phi.ravel().copy()
    delta, sign = np.zeros(want.size), np.zeros(want.size)
    if ndim > 1 and scale <= 1:  # stores delta; needs cells within the width, and two axes
        m0 = ls.mass(width, 1e-3)
        ls.mpls(dt, width, 1e-3, m0, count=1)
        oracle.lib.orc_mpls_euler(ndim, *n, *h, dt, width, 1e-3, 1, m0, types, vals, want, 1, delta.ctypes.data)
        want = ls.phi().ravel().copy()
    ls.find_sign(width)
    oracle.lib.orc_find_sign(want.size, want, width, sign)
    ls.redistance(dt, rdt, steps)
    oracle.lib.orc_redistance_rk3(ndim, *n, *h, dt, rdt, sign, delta, types, vals, want, steps)
    return ls.phi().ravel(), want


@pytest.mark.parametrize("bc", BCS, ids=lambda b: "-".join(x[:3] for x in b[:4]))
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_redistance_matches_oracle(oracle, n, bc):
    got, want = _run(oracle, n, bc, 1.0, 2)
    assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("scale", [1e-30, 1e15, 1e26, 1e60])
def test_redistance_weights_at_any_magnitude(oracle, scale):
    """second differences of 1e-3 scale: their fourth powers reach 1e228"""
    got, want = _run(oracle, (30, 41, 1), ["neumann"] * 6, scale, 1)
    assert np.isfinite(want).all()
    assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
