"""The fused WENO5 TVD-RK3 stage (k_rk3_fused) against the oracle at the edges
of its tiles: rows of 62, 63 and 64 cells, several short rows a wavefront (30,
31 and 32 cells and fewer), marches that end early, 3-D row tiles of 6, 7 and 8
and of several short rows, and every boundary condition, mixed over
the sides (Dirichlet sides take the separate ghost kernels).

Bar: 1e-13 of the largest value after two steps; a face value is formed from
about 60 FP64 operations in another order than the oracle's, and enters the
level set times dt u / h <= 0.2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.pyoracle import Oracle
from scihpc_amd import LevelSet, padded_shape
from scihpc_amd._capi import BC_CODES

SHAPES = [(3, 4, 1), (5, 62, 1), (33, 63, 1), (20, 64, 1), (7, 127, 1), (900, 190, 1), (6, 6, 62), (9, 7, 64), (13, 8, 5),
          (20, 15, 126), (100, 30, 1), (7, 31, 1), (50, 32, 1), (700, 20, 1), (9, 15, 31), (5, 16, 31), (8, 23, 20),
          (12, 24, 20), (6, 50, 9), (5, 3, 30)]
BCS = [["neumann"] * 6, ["periodic"] * 6, ["no_slip", "slip", "neumann", "no_slip", "slip", "neumann"],
       ["dirichlet", "neumann", "slip", "dirichlet", "neumann", "dirichlet"]]


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


@pytest.mark.parametrize("bc", BCS, ids=lambda b: "-".join(x[:3] for x in b[:4]))
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_fused_stage_matches_oracle(oracle, n, bc):
    ndim = 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 0.8 / n[1], 1.1 / n[2])
    shp = padded_shape(ndim, *n)
    rng = np.random.default_rng(sum(n))
    phi = rng.standard_normal(shp)
    vel = [rng.standard_normal(shp) for _ in range(3)]
    vals = np.linspace(-0.3, 0.4, 6)
    dt = 0.05 * min(h[:ndim])
    print(f"fused stage {n} {bc}", flush=True)
    ls = LevelSet(ndim, *n, *h, bc, list(vals))
    ls.set_phi(phi)
    ls.set_velocity(*vel)
    ls.tvd_rk3(dt, 2)
    want = phi.ravel().copy()
    tmp = [np.zeros(want.size) for _ in range(3)]
    types = np.array([BC_CODES[b] for b in bc], np.int32)
    oracle.lib.orc_tvd_rk3_weno(ndim, *n, *h, dt, types, vals, want, *[a.ravel() for a in vel], *tmp, 2)
    inner = tuple(slice(3, -3) if a < ndim else slice(None) for a in range(3))
    got, want = ls.phi(), want.reshape(shp)
    big = np.abs(want[inner]).max()
    for a in range(ndim):  # every line through the interior, its ghosts included
        at = tuple(slice(None) if d == a else s for d, s in enumerate(inner))
        assert np.abs(got[at] - want[at]).max() < 1e-13 * big


@pytest.mark.parametrize("n", [(33, 63, 1), (6, 7, 13)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("kind,scale", [("steps", 1e60), ("steps", 1e100), ("steps", 1e140), ("random", 2e152)])
def test_fused_stage_at_any_magnitude(oracle, n, kind, scale):
    """fields of two values, whose weights next to a flat stencil are their
    differences squared over 1e-8, and fields whose squares nearly overflow
    (up to 13 (4 s)^2 + 3 (8 s)^2 = 1.6e307 for s = 2e152; periodic, as a flat
    stencil at a wall makes the weights themselves overflow from s = 1e149 on):
    finite where the normalised weights are.  Same bar."""
    ndim = 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 0.8 / n[1], 1.1 / n[2])
    shp = padded_shape(ndim, *n)
    rng = np.random.default_rng(sum(n))
    phi = scale * (np.where(rng.random(shp) < 0.5, 1.0, -1.0) if kind == "steps" else rng.uniform(-1, 1, shp))
    vel = [rng.standard_normal(shp) for _ in range(3)]
    dt = 0.05 * min(h[:ndim])
    print(f"fused stage {n} {kind} {scale:g}", flush=True)
    bc = "periodic" if kind == "random" else "neumann"
    ls = LevelSet(ndim, *n, *h, [bc] * 6)
    ls.set_phi(phi)
    ls.set_velocity(*vel)
    ls.tvd_rk3(dt, 2)
    want = phi.ravel().copy()
    tmp = [np.zeros(want.size) for _ in range(3)]
    types = np.full(6, BC_CODES[bc], np.int32)
    oracle.lib.orc_tvd_rk3_weno(ndim, *n, *h, dt, types, np.zeros(6), want, *[a.ravel() for a in vel], *tmp, 2)
    inner = tuple(slice(3, -3) if a < ndim else slice(None) for a in range(3))
    got, want = ls.phi()[inner], want.reshape(shp)[inner]
    assert np.isfinite(want).all()
    assert np.abs(got / scale - want / scale).max() < 1e-13 * np.abs(want / scale).max()


@pytest.mark.parametrize("bc", BCS, ids=lambda b: "-".join(x[:3] for x in b[:4]))
@pytest.mark.parametrize("n", [(3, 4, 1), (33, 63, 1), (40, 1, 1), (6, 7, 5)], ids=lambda n: "x".join(map(str, n)))
def test_uccd_stage_fills_its_ghosts(oracle, n, bc):
    """k_uccd_stage's ghosts: the oracle's bits, corners too (next to a
    Dirichlet side bc_line fills them, whose U h + F the compiler may round
    once: values of zero there)"""
    ndim = 1 if n[1] == 1 else 2 if n[2] == 1 else 3
    h = (1.0 / n[0], 0.8 / n[1], 1.1 / n[2])
    shp = padded_shape(ndim, *n)
    rng = np.random.default_rng(sum(n))
    phi = rng.standard_normal(shp)
    vel = [rng.standard_normal(shp) for _ in range(3)]
    vals = np.zeros(6) if "dirichlet" in bc else np.linspace(-0.3, 0.4, 6)
    dt = 0.05 * min(h[:ndim])
    print(f"uccd stage {n} {bc}", flush=True)
    ls = LevelSet(ndim, *n, *h, bc, list(vals))
    ls.set_phi(phi)
    ls.set_velocity(*vel)
    ls.set_scheme("uccd")
    ls.tvd_rk3(dt, 2)
    want = phi.ravel().copy()
    types = np.array([BC_CODES[b] for b in bc], np.int32)
    oracle.lib.orc_tvd_rk3_uccd(ndim, *n, *h, dt, types, vals, want, *[a.ravel() for a in vel], 2)
    np.testing.assert_array_equal(ls.phi().ravel(), want)
