"""The face kernels' short forms (the limiter's common case, the Rusanov flux
without the rotation's zero products, the square root without its special
cases) hand every state outside their range to the reference's operations:
FVTD outputs are bitwise the oracle's on states that mix both -- dry cells,
depths and velocities at the edges of the short forms, signed zeros, Inf and
NaN -- at grid sizes around the tiles' edges."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import FVTD_KEYS, describe_diff, fvtd_view, same_bits

pytestmark = pytest.mark.gpu

KINDS = {
    # depths that make the limiter act, and dry cells
    "dry": ([0.0, 1e-7, 1e-6, 1e-3, 1.0], [0.0, 0.5, -2.0]),
    # depths below and above the square root's and the depths' ranges
    "range": ([1e-310, 1e-181, 1e-180, 1.0, 1e100, 1e154], [0.0, 1e-30, 1.0]),
    # velocities of either zero, subnormal and huge
    "zeros": ([0.5, 1.0, 2.0], [0.0, -0.0, 5e-324, -5e-324, 1e-310, 1e-160, 1e120]),
    # a few cells that are not finite
    "nonfinite": ([1.0, 1.5, 2.0], [0.1, -0.2, 0.0]),
}


def state(kind, n, ny, seed):
    rng = np.random.default_rng(seed)
    hs, us = KINDS[kind]
    U = np.empty((ny, n, 3))
    smooth = 1.0 + 0.05 * np.sin(np.arange(n) / 3.0)[None, :] * np.cos(np.arange(ny) / 4.0)[:, None]
    odd = rng.uniform(size=(ny, n)) < 0.3
    U[..., 0] = np.where(odd, rng.choice(hs, (ny, n)), smooth)
    for v in (1, 2):
        with np.errstate(over="ignore", under="ignore", invalid="ignore"):
            U[..., v] = U[..., 0] * np.where(odd, rng.choice(us, (ny, n)), 0.1 * smooth)
    if kind == "nonfinite":
        for v, x in ((0, np.inf), (1, np.nan), (2, np.inf), (1, -np.inf)):
            U[rng.integers(0, ny), rng.integers(0, n), v] = x
    return P.Problem(n, U, kind=kind, ny=ny)


# shape -1: the launch's own choice, two lanes per cell at these sizes
@pytest.mark.parametrize("shape", [0, 1, -1])
@pytest.mark.parametrize("size", [(17, 31), (33, 32), (48, 15)])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_fvtd_matches_oracle(kind, size, shape):
    p = state(kind, *size, seed=7)
    ref = Oracle(p).fvtd()
    s = swm.Solver.from_problem(p)
    s.set_tile_shape(shape)
    got = s.fvtd()
    for k in FVTD_KEYS:
        a, b = fvtd_view(got, k), fvtd_view(ref, k)
        assert same_bits(a, b), f"{kind} {size} {k}: {describe_diff(a, b)}"


@pytest.mark.parametrize("recfix", [1, 2])
@pytest.mark.parametrize("size", [(3, 5), (15, 17), (31, 48)])
def test_two_lanes_per_cell_with_the_shock_fix(size, recfix):
    p = state("dry", *size, seed=11)
    ref = Oracle(p, recfix=recfix).fvtd()
    s = swm.Solver.from_problem(p, recfix=recfix)
    got = s.fvtd()
    for k in FVTD_KEYS:
        a, b = fvtd_view(got, k), fvtd_view(ref, k)
        assert same_bits(a, b), f"{size} fix {recfix} {k}: {describe_diff(a, b)}"
