"""The one-workgroup coarse cycle (k_block_vcycle) at the shapes where it can
go wrong: a single (coarsest) level, odd sizes (a pair with no odd cell),
ragged patches, factor-3 levels, every patch height, a large coarsest
matrix, 2-D and 3-D, zero and non-zero initial iterates, unequal sweep
counts; and the 3-D tiles (k_pre3d, k_post3d) above it, whole and ragged.

Bars: FP64 iterates within 1e-10 relative of the oracle's red-black cycle
(both sum five or seven terms in FP64; the cycles amplify that by far less
than 1e5), FP32 within 2e-5 (about 100 ulp of FP32 over the cycle's 40
stages), as for the tiled kernels.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.pyoracle import Oracle
from scihpc_amd import PREC_MIXED, Multigrid


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


# shape, bc, variable
CASES = [
    ((5, 7, 1), "neumann", True),      # the coarsest level alone
    ((10, 14, 1), "dirichlet", False),
    ((30, 42, 1), "neumann", True),    # 15 x 21 -> 5 x 7 by 3
    ((26, 38, 1), "neumann", True),    # 13 x 19 coarsest, odd rows of pairs
    ((45, 75, 1), "neumann", True),    # odd top level, factor 3, 375 unknowns
    ((45, 75, 1), "dirichlet", False),
    ((58, 62, 1), "neumann", True),    # two-row patches
    ((58, 66, 1), "dirichlet", False),
    ((132, 156, 1), "neumann", True),  # 66 x 78 in the block in FP32
    ((120, 228, 1), "neumann", True),  # four-row patches, ragged, in FP32
    ((128, 256, 1), "neumann", False),
    ((4, 6, 5), "neumann", True),
    ((12, 10, 14), "neumann", True),
    ((18, 18, 18), "neumann", True),   # 9^3 coarsest
    ((16, 16, 16), "dirichlet", False),
    ((30, 18, 24), "neumann", True),
    ((32, 32, 32), "neumann", True),   # 3-D tiles on level 0 (first cycle only: from zero)
    ((64, 32, 48), "dirichlet", False),
    ((72, 60, 48), "neumann", True),   # also on 36 x 30 x 24: ragged in x and y
]


def _pair(oracle, case):
    (nx, ny, nz), bc, var = case
    ndim = 2 if nz == 1 else 3
    h = (1.0 / nx, 1.1 / ny, 0.9 / nz)
    g, o = Multigrid(ndim, nx, ny, nz, *h, bc), oracle.mg(ndim, nx, ny, nz, *h, bc)
    rng = np.random.default_rng(nx * 1000 + ny)
    n = nx * ny * nz
    if var:
        rho = np.exp(rng.uniform(0, np.log(1000.0), n))
        g.set_density(rho)
        o.set_rho(rho)
    b = rng.standard_normal(n)
    return g, o, b - b.mean() if bc == "neumann" else b


def _ids(c):
    return "x".join(str(v) for v in c[0]) + "-" + c[1] + ("-var" if c[2] else "")


@pytest.mark.parametrize("nu", [(2, 2), (1, 2), (0, 1), (2, 0)], ids=lambda v: f"V{v[0]}{v[1]}")
@pytest.mark.parametrize("case", CASES, ids=_ids)
def test_block_cycle_matches_oracle(oracle, case, nu):
    g, o, b = _pair(oracle, case)
    print(f"block cycle {case} {nu}", flush=True)
    g.set_rhs(b)
    g.set_sol(np.zeros_like(b))
    o.vec(0, "rhs")[:] = b
    o.vec(0, "sol")[:] = 0
    for _ in range(2):
        g.v_cycle(*nu)
        oracle.lib.orc_mg_vcycle_rb(o.h, *nu)
        x = o.vec(0, "sol")
        e = np.linalg.norm(g.sol(0) - x) / np.linalg.norm(x)
        assert e < 1e-10, e


@pytest.mark.parametrize("case", CASES, ids=_ids)
def test_block_cycle_fp32_matches_oracle(oracle, case):
    g, o, b = _pair(oracle, case)
    print(f"block cycle FP32 {case}", flush=True)
    g.set_rhs(b)
    g.solve(rel_tol=1e-30, max_cycles=1, precision=PREC_MIXED, accel=0)
    o.vec(0, "rhs")[:] = b
    o.vec(0, "sol")[:] = 0
    oracle.lib.orc_mg_vcycle_rb(o.h, 2, 2)
    x = o.vec(0, "sol").copy()
    if case[1] == "neumann":
        x -= x.mean()
    e = np.linalg.norm(g.sol(0) - x) / np.linalg.norm(x)
    assert e < 2e-5, e
