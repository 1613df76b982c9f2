"""Stage combinations of the explicit schemes that take the last FVTD's fluxes
as they are, against the oracle and against the same steps with the derivatives
stored first (which recording events asks for), bitwise: small launches with
and without bathymetry and the well-balanced state, large ones without, and
fluxes below the range of the shared reciprocal."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import describe_diff, same_bits

pytestmark = pytest.mark.gpu


def tiny_momenta(n, ny):
    rng = np.random.default_rng(4)
    U = np.ones((ny, n, 3))
    U[..., 1:] = 1e-140 * rng.normal(size=(ny, n, 2))
    U[ny // 2:, :, 1:] = 0.0
    return P.Problem(n, U, kind="tiny", ny=ny)


def random_state(n, ny):
    rng = np.random.default_rng(n)
    U = np.empty((ny, n, 3))
    U[..., 0] = 1.0 + 0.2 * rng.uniform(-1, 1, (ny, n))
    U[..., 1:] = 0.2 * rng.normal(size=(ny, n, 2))
    return P.Problem(n, U, kind="random", ny=ny)


CASES = {
    "tiny33x20": lambda: tiny_momenta(33, 20),
    "lake_bumps40": lambda: P.lake_bumps(40, 4),
    "lake_flag1_no_wb24": lambda: P.lake_flag1(24, False),
    "random256x3": lambda: random_state(256, 3),
}


@pytest.mark.parametrize("scheme", [1, 2, 3, 4])
@pytest.mark.parametrize("case", sorted(CASES))
def test_small(case, scheme):
    p = CASES[case]()
    s = swm.Solver.from_problem(p)
    s.set_timescheme(scheme)
    dts, _, _ = s.run_steps(3)
    o = Oracle(p, scheme)
    for dt in dts:
        o.step(dt)
    assert same_bits(s.download(), o.get_U()), describe_diff(s.download(), o.get_U())


@pytest.mark.parametrize("scheme", [2, 3, 4])
def test_large(scheme):
    p = random_state(1100, 1030)
    out = []
    for events in (False, True):
        s = swm.Solver.from_problem(p)
        s.set_timescheme(scheme)
        s.profile(events)
        s.run_steps(2)
        out.append(s.download())
    assert same_bits(*out)
