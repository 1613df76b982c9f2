"""Waits of the one-launch Patankar solve that run out, forced from the host by
a limit of no polls, under which every kernel still ends by itself: the step is
run again and stays the oracle's bit for bit, the solve rests for some batches
and is used again after them, and solves that never wait do not rest."""
from __future__ import annotations

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import describe_diff, same_bits

pytestmark = pytest.mark.gpu


def random_state(nx, ny, seed):
    rng = np.random.default_rng(seed)
    U = np.empty((ny, nx, 3))
    U[..., 0] = 1.0 + 0.3 * rng.uniform(-1, 1, (ny, nx))
    U[..., 1:] = U[..., :1] * rng.normal(0, 0.3, (ny, nx, 2))
    return P.Problem(nx, U, kind="random", ny=ny)


def until_solved(s, o):
    """Steps of one batch each until the solve is used again; returns their number."""
    before = s.solve_stats()["steps"]
    for k in range(200):
        assert s.run_steps(1)[0][0] == o.timestep()[0]
        o.step(o.timestep()[0])
        if s.solve_stats()["steps"] > before:
            return k
    raise AssertionError("the solve is not used again")


@pytest.mark.parametrize("size", [(90, 70), (113, 20)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_lost_wait_and_recovery(size):
    p = random_state(*size, 5)
    s, o = swm.Solver.from_problem(p), Oracle(p)
    assert until_solved(s, o) == 0
    rests = []
    for n in (1, 2, 3):
        # six steps on the stream: the first loses its wait, the others end early
        s.debug_solve_polls(0)
        dts, _, _ = s.run_steps(1 if n == 2 else 6)
        s.debug_solve_polls(-1)
        for dt in dts:
            assert o.timestep()[0] == dt
            o.step(dt)
        assert s.solve_stats()["lost"] == n
        assert s.execution_stats()["redone_steps"] >= n
        rests.append(s.solve_stats()["resting"])
        assert until_solved(s, o) == rests[-1]
        assert s.solve_stats()["resting"] == 0
    assert 0 < rests[0] < rests[1]
    for _ in range(3):  # and in use from here on
        assert until_solved(s, o) == 0
    assert s.execution_stats()["redone_steps"] >= 3
    U, V = s.download(), o.get_U()
    assert same_bits(U, V), describe_diff(U, V)


def test_solves_without_waits_do_not_rest():
    p = random_state(40, 30, 6)
    s, o = swm.Solver.from_problem(p), Oracle(p)
    s.debug_solve_polls(0)
    for k in range(3):
        assert until_solved(s, o) == 0
    assert s.solve_stats() == {"steps": 3, "lost": 0, "resting": 0}
    assert same_bits(s.download(), o.get_U())
