"""State transfers through the pinned ring: bitwise round trips at sizes around
its chunks, its slots and the largest upload it takes, with ghost layers; the
end of a step on grids around the largest it commits in one launch; and two
threads with solvers of their own, which share the ring and take turns at the
one-launch solves."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import same_bits

pytestmark = pytest.mark.gpu

CHUNK = (1 << 19) // 24  # cells of a 512 KB chunk


def state(nx, ny, seed):
    rng = np.random.default_rng(seed)
    U = np.empty((ny, nx, 3))
    U[..., 0] = 1.0 + 0.2 * rng.uniform(-1, 1, (ny, nx))
    U[..., 1:] = 0.1 * rng.normal(size=(ny, nx, 2))
    return U


@pytest.mark.parametrize("ghosts", [0, 3])
@pytest.mark.parametrize("size", [(3, 3), (CHUNK // 3, 3), (CHUNK // 3 + 1, 3), (4 * CHUNK, 4),
                                  (4 * CHUNK + 1, 3), (409, 427), (410, 427), (1031, 700)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_round_trip(size, ghosts):
    nx, ny = size
    U = state(nx, ny, nx)
    s = swm.Solver.from_problem(P.Problem(nx, state(nx, ny, 1), kind="random", ny=ny))
    ext = np.full((ny + 2 * ghosts, nx + 2 * ghosts, 3), np.nan)
    ext[ghosts:ghosts + ny, ghosts:ghosts + nx] = U
    s.upload(ext, ghosts)
    assert same_bits(s.download(), U)


# cells: 63, 64, 65, 4092, 4096, 4160
@pytest.mark.parametrize("size", [(9, 7), (8, 8), (13, 5), (62, 66), (64, 64), (64, 65)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("scheme", [2, 5])
def test_step_end(size, scheme):
    nx, ny = size
    p = P.Problem(nx, state(nx, ny, 3), kind="random", ny=ny)
    s = swm.Solver.from_problem(p)
    s.set_timescheme(scheme)
    dts, _, _ = s.run_steps(3)
    o = Oracle(p, scheme)
    for k in range(3):
        assert o.timestep()[0] == dts[k]
        o.step(dts[k])
    assert same_bits(s.download(), o.get_U())


def test_two_threads():
    ps = [P.Problem(90, state(90, 70, 5), kind="random", ny=70),
          P.Problem(500, state(500, 400, 6), kind="random", ny=400)]

    def work(p):
        s = swm.Solver.from_problem(p)
        out = []
        for _ in range(4):
            s.upload(p.U0)
            s.run_steps(2)
            out.append(s.download())
        return out

    alone = [work(p)[0] for p in ps]
    got = [None, None]

    def run(i):
        got[i] = work(ps[i])

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in range(2):
        assert all(same_bits(U, alone[i]) for U in got[i])
