"""That the solve in one launch is what ran where it is meant to: every tile size
and every number of rows per thread, on first and later steps, several launches
where the systems do not fit at once, two threads taking turns; and the momenta
around rows outside its short form."""
from __future__ import annotations

import threading

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


# one block at 1, 2, 4 rows per thread; tiles of 2, 3, 5, 8 and 11
SIZES = [(32, 16), (32, 32), (64, 32), (49, 73), (257, 250), (419, 418), (700, 650), (1024, 1000)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_used_from_the_first_step(size):
    p = random_state(*size, 11)
    s = swm.Solver.from_problem(p)
    s.run_steps(3)
    st = s.execution_stats()
    assert s.solve_stats() == {"steps": 3, "lost": 0, "resting": 0}
    assert st["speculative_steps"] == 3 and st["redone_steps"] == 0
    assert st["graph_captures"] == 0  # replay gains nothing: only where it is asked for
    t = swm.Solver.from_problem(p)
    t.set_execution(0, -2)
    t.run_steps(3)
    assert t.solve_stats()["steps"] == 0
    assert same_bits(s.download(), t.download())


def test_cut_into_launches():
    """Ten grids of 12 tiles and more: three systems each do not fit at once."""
    eng = swm.Engine()
    ids = [eng.submit(random_state(190 + 3 * k, 200 - 2 * k, k), 2) for k in range(10)]
    eng.profile(True)
    while eng.run(4)[0]:
        pass
    eng.profile(False)
    steps = eng.solve_stats()["steps"]
    assert steps == 2 and eng.solve_stats()["lost"] == 0 and len(ids) == 10
    launches = eng.profile_read()["jacobi_sweep"][1]
    assert launches > 5 * steps  # more than one a correction


def test_two_threads_take_turns():
    ps = [random_state(90, 70, 5), random_state(500, 400, 6)]
    got, used = [None, None], [0, 0]

    def run(i):
        s = swm.Solver.from_problem(ps[i])
        for _ in range(6):
            s.run_steps(1)
        got[i], used[i] = s.download(), s.solve_stats()["steps"]
        assert s.solve_stats()["lost"] == 0

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert sum(used) > 0
    for p, U in zip(ps, got):
        s = swm.Solver.from_problem(p)
        s.set_execution(0, -2)
        s.run_steps(6)
        assert same_bits(U, s.download())


@pytest.mark.parametrize("low", [0.0, 1e-65])
@pytest.mark.parametrize("n", [20, 44, 90, 300])
def test_momenta_around_rows_out_of_the_short_form(n, low):
    """Bit for bit wherever they are numbers (NaN where the dry bed makes them so, on
    20^2 everywhere)."""
    p = P.dam_break(n, 1, dry=low)
    s, o = swm.Solver.from_problem(p), Oracle(p)
    dts, _, _ = s.run_steps(1)
    o.step(dts[0])
    assert s.solve_stats()["steps"] == 1
    U, V = s.download(), o.get_U()
    assert np.isfinite(V[..., 1:]).any() == (n > 20)
    assert same_bits(U, V), describe_diff(U, V)
