"""TimeStep's fold with 256 threads and with 1024, at the number of partial maxima
where the one gives way to the other and at the smallest grids, bitwise against
the oracle -- also with a NaN speed, which makes the fold depend on its order."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import same_bits

pytestmark = pytest.mark.gpu


# 2048 partial maxima are 524,288 cells
@pytest.mark.parametrize("nan", [False, True])
@pytest.mark.parametrize("size", [(3, 3), (16, 16), (17, 16), (1024, 512), (1025, 512)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_timestep(size, nan):
    nx, ny = size
    rng = np.random.default_rng(nx + ny)
    U = np.empty((ny, nx, 3))
    U[..., 0] = 1.0 + 0.3 * rng.uniform(-1, 1, (ny, nx))
    U[..., 1:] = rng.normal(0, 0.3, (ny, nx, 2))
    if nan:
        U[ny // 2, nx // 2, 1] = np.nan
        U[0, 1, 2] = np.nan
    p = P.Problem(nx, U, kind="random", ny=ny)
    s, o = swm.Solver.from_problem(p), Oracle(p)
    assert same_bits(s.timestep(), o.timestep())
