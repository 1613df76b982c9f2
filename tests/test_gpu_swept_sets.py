"""Job sets with a launch per sweep, which the one-launch solve takes over where
it can: the autotuner really tunes there, leaves a caller's records alone, and a
step with too few sweeps is run again (stage minima keep the solve in one launch
off); and one engine whose solved and swept grids step together."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import describe_diff, same_bits

pytestmark = pytest.mark.gpu

TIMED = 2 * (2 + 4)  # tuning steps: two rounds over the shapes and over (graph, margin)


def swept(p):
    s = swm.Solver.from_problem(p)
    s.track_stage_min(True)
    return s


def test_autotuner_tunes_a_swept_set():
    p = P.vortex(96, 7)
    s = swept(p)
    before = s.status_reads()
    s.run_steps(1 + TIMED + 4)
    # a read a step while it tunes; batches afterwards
    assert s.status_reads() - before > TIMED
    before, redone = s.status_reads(), s.execution_stats()["redone_steps"]
    s.run_steps(16)
    if s.execution_stats()["redone_steps"] == redone:
        assert s.status_reads() - before <= 2
    st = s.execution_stats()
    assert st["graph_captures"] >= 2  # margins 1 and 2
    assert st["graph"] in (0, 1) and st["margin"] in (1, 2) and s.tile_shape()[0] in (0, 1)
    assert s.solve_stats()["steps"] == 0
    o = Oracle(p)
    o.run(1 + TIMED + 20)
    assert same_bits(s.download(), o.get_U())


def test_tuner_leaves_unread_records_of_a_swept_set():
    p = P.vortex(48, 5)
    s = swept(p)
    s.profile(True)
    s.run_steps(1)  # 5 launches of each face kernel
    s.profile(False)
    before = s.status_reads()
    s.run_steps(TIMED + 8)
    assert s.status_reads() - before > TIMED
    rec = s.profile_read()
    assert rec["fvtd_x"][1] == 5 and rec["fvtd_y"][1] == 5 and rec["fvtd_x"][0] > 0.
    o = Oracle(p)
    o.run(TIMED + 9)
    assert same_bits(s.download(), o.get_U())


@pytest.mark.parametrize("graph", [0, 1])
def test_underpredicted_swept_step_is_redone(graph):
    p = P.vortex(32, 4)
    s = swept(p)
    s.set_execution(graph, 0)
    s.set_jacobi_limits(2, 1e-16)  # predicts 2 sweeps
    s.run_steps(1)
    s.set_jacobi_limits(1000, 1e-16)
    s.run_steps(2)
    assert s.execution_stats()["redone_steps"] >= 1 and s.solve_stats()["steps"] == 0
    o = Oracle(p)
    for k in range(3):
        o.set_jacobi_limits(*((2, 1e-16) if k == 0 else (1000, 1e-16)))
        o.step(o.timestep()[0])
    assert same_bits(s.download(), o.get_U())


def random_state(nx, ny, seed, amp):
    rng = np.random.default_rng(seed)
    U = np.empty((ny, nx, 3))
    U[..., 0] = 1.0 + amp * rng.uniform(-1, 1, (ny, nx))
    U[..., 1:] = U[..., :1] * rng.normal(0, amp, (ny, nx, 2))
    return P.Problem(nx, U, kind="random", ny=ny)


def plain(p, steps):
    s = swm.Solver.from_problem(p)
    s.set_execution(0, -2)  # a launch per sweep, each looked at
    s.run_steps(steps)
    return s.download()


def test_solved_and_swept_grids_in_one_engine():
    """A grid with more tiles than the device holds blocks beside one of one block,
    one of several and one with bathymetry, leaving at different steps; and a swept
    grid whose sweeps grow, so that its step alone is run again."""
    jobs = [(random_state(1190, 1010, 1, 0.01), 4), (random_state(40, 30, 2, 0.3), 2),
            (random_state(150, 131, 3, 0.3), 5), (P.lake_bumps(70, 4), 3)]
    # at rest in the first step but for a pulse: few sweeps first, more later
    calm = random_state(1190, 1010, 5, 0.0)
    calm.U0[500:510, 500:510, 0] += 0.3
    for big in (jobs[0][0], calm):
        eng = swm.Engine()
        eng.set_execution(0, -1)
        todo = [(big, 4)] + jobs[1:]
        ids = [eng.submit(p, k) for p, k in todo]
        while eng.run(4)[0]:
            pass
        assert eng.solve_stats()["steps"] > 0 and eng.solve_stats()["lost"] == 0
        for (p, k), j in zip(todo, ids):
            U, V = eng.fetch(j), plain(p, k)
            assert same_bits(U, V), (p.n, describe_diff(U, V))
