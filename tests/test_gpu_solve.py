"""The Patankar solve in one launch (k_solve) against the oracle, bitwise with
its sweep counts: one block and several, at the sizes where the number of
blocks or of rows per thread changes, on grids wider than a block's rows and
narrower than a wave; several solves cut into launches; and its ways out --
a sweep limit and a stop decision left open."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import describe_diff, same_bits

pytestmark = pytest.mark.gpu


def random_state(n, ny, seed, amp=0.3):
    rng = np.random.default_rng(seed)
    U = np.empty((ny, n, 3))
    U[..., 0] = 1.0 + amp * rng.uniform(-1, 1, (ny, n))
    U[..., 1] = U[..., 0] * rng.normal(0, 0.3, (ny, n))
    U[..., 2] = U[..., 0] * rng.normal(0, 0.3, (ny, n))
    return P.Problem(n, U, kind="random", ny=ny)


# nx, ny, steps: 512, 1024 and 2048 cells are the most that one block takes at
# 1, 2 and 4 rows per thread; from 2049 on the tiles of a system share a
# solve: tiles of at most 56 x 8, 16, 32, 56 and 80 cells (full ones and one
# cell more; thinner than the 4 cells of halo; a grid thinner than its halo)
SIZES = [(3, 3, 3), (32, 16, 3), (27, 19, 3), (32, 32, 2), (41, 25, 2), (64, 32, 2), (3, 683, 2),
         (683, 3, 2), (1500, 4, 2), (48, 48, 2), (49, 73, 2), (56, 40, 2), (57, 41, 2),
         (101, 67, 2), (112, 80, 2), (192, 193, 1), (240, 238, 1), (241, 239, 1), (419, 418, 1),
         (517, 513, 1)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_solve_matches_oracle(size):
    nx, ny, steps = size
    p = random_state(nx, ny, nx + ny)
    s = swm.Solver.from_problem(p)
    o = Oracle(p)
    dts, sweeps, _ = s.run_steps(steps)
    for k in range(steps):
        dt, _, _ = o.timestep()
        it = o.step(dt)
        it = it[0] if isinstance(it, tuple) else it
        assert dt == dts[k]
        assert list(sweeps[k]) == list(it)[:13]
    assert s.execution_stats()["redone_steps"] == 0
    assert same_bits(s.download(), o.get_U()), describe_diff(s.download(), o.get_U())


@pytest.mark.parametrize("low", [0.0, 1e-65])
@pytest.mark.parametrize("n", [20, 44, 90, 300])
def test_rows_out_of_the_short_form_range(n, low):
    """Depths of zero and below 2^-200 around a dam: their blocks take the full
    form of the sweep, the others the short one.  (The momenta there are NaN.)"""
    p = P.dam_break(n, 1, dry=low)
    s = swm.Solver.from_problem(p)
    o = Oracle(p)
    dts, sweeps, _ = s.run_steps(1)
    it = o.step(dts[0])
    it = it[0] if isinstance(it, tuple) else it
    assert list(sweeps[0]) == list(it)[:13]
    assert s.execution_stats()["redone_steps"] == 0
    U, V = s.download(), o.get_U()
    assert same_bits(U[..., 0], V[..., 0])
    assert (np.isnan(U) == np.isnan(V)).all()


@pytest.mark.parametrize("scheme", [6, 7])
@pytest.mark.parametrize("size", [(40, 40), (90, 70)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_two_node_schemes(size, scheme):
    p = random_state(*size, 3)
    s = swm.Solver.from_problem(p)
    s.set_timescheme(scheme)
    s.set_hp_association(swm.HP_BY_NODE)
    dts, _, _ = s.run_steps(2)
    o = Oracle(p, scheme, hp_by_node=True)
    for k in range(2):
        assert o.timestep()[0] == dts[k]
        o.step(dts[k])
    assert same_bits(s.download(), o.get_U())


def test_several_launches_match_plain_solvers():
    """More blocks than the device holds at once: the engine cuts the solves
    into launches; every job is bitwise the plain solver's."""
    jobs = [(random_state(190 + 3 * k, 200 - 2 * k, k), 2) for k in range(10)]
    jobs += [(random_state(20 + k, 30, 50 + k), 3) for k in range(3)]
    eng = swm.Engine()
    ids = [eng.submit(p, k) for p, k in jobs]
    while eng.run(4)[0]:
        pass
    for (p, k), j in zip(jobs, ids):
        s = swm.Solver.from_problem(p)
        s.set_execution(0, -2)  # a launch per sweep
        s.run_steps(k)
        assert same_bits(eng.fetch(j), s.download())


@pytest.mark.parametrize("size", [(1027, 1023), (1023, 1024)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_grouped_residual_sums(size):
    """The last grid with a residual sum per 256 cells and the first, ragged,
    with one per 1024: sweeps launched one by one, against the solve in one
    launch."""
    p = random_state(*size, 7)
    a, b = swm.Solver.from_problem(p), swm.Solver.from_problem(p)
    b.set_execution(0, -2)
    ra, rb = a.run_steps(1), b.run_steps(1)
    assert ra[0] == rb[0] and (ra[1] == rb[1]).all()
    assert same_bits(a.download(), b.download())


@pytest.mark.parametrize("scheme,wb", [(5, False), (5, True), (7, False)])
@pytest.mark.parametrize("size", [(1000, 900), (1100, 1030)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_assembly_of_large_grids_from_the_fluxes(size, scheme, wb):
    """Without bathymetry the assembly takes the fluxes as they are, before the
    one-launch solve and before launches per sweep; recording events keeps the
    update before it."""
    p = random_state(*size, 9)
    if wb:
        p.wellbalanced, p.Uwb = True, random_state(*size, 10, 0.01).U0
    out = []
    for events in (False, True):
        s = swm.Solver.from_problem(p)
        s.set_timescheme(scheme)
        s.set_hp_association(swm.HP_BY_NODE)
        s.profile(events)
        dts, sweeps, _ = s.run_steps(2)
        out.append((s.download(), dts, sweeps))
    assert (out[0][1] == out[1][1]).all() and (out[0][2] == out[1][2]).all()
    assert same_bits(out[0][0], out[1][0])


@pytest.mark.parametrize("size", [(32, 32), (80, 80)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_open_decision_is_taken_by_the_sequential_sum(size):
    """A uniform depth 1 at rest with the tolerance 1: the initial residual is
    exactly the tolerance, inside the certified window, so the step is run
    again and the sequential sum decides."""
    n, ny = size
    U = np.zeros((ny, n, 3))
    U[..., 0] = 1.0
    p = P.Problem(n, U, kind="uniform", ny=ny)
    s = swm.Solver.from_problem(p)
    s.set_jacobi_limits(1000, 1.0)
    dts, sweeps, _ = s.run_steps(1)
    assert s.execution_stats()["redone_steps"] == 1
    assert s.ambiguous_decisions() >= 13
    o = Oracle(p)
    o.set_jacobi_limits(1000, 1.0)
    dt, _, _ = o.timestep()
    o.step(dt)
    assert same_bits(s.download(), o.get_U())


def test_sweep_limit_without_convergence():
    """max_iter below what the solves need: they stop there, counted as not
    converged, as the oracle's do."""
    p = P.vortex(70, 5)
    s = swm.Solver.from_problem(p)
    s.set_jacobi_limits(3, 1e-16)
    dts, sweeps, nonconv = s.run_steps(2)
    assert nonconv == 26 and (sweeps == 3).all()
    o = Oracle(p)
    o.set_jacobi_limits(3, 1e-16)
    for k in range(2):
        o.step(dts[k])
    assert same_bits(s.download(), o.get_U())
