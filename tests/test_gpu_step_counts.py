"""A batch of an engine launches no more steps than the running job with most of
them left has to go: what lies behind a job's last step is not computed."""
from __future__ import annotations

import pytest

import problems as P
import swm
from oracle_api import Oracle
from parity_util import same_bits

pytestmark = pytest.mark.gpu

# launches of one step: assemblies (one per correction) or stage combinations
CATEGORY = {5: ("patankar_assemble", 5), 7: ("patankar_assemble", 2), 2: ("momentum", 5)}


@pytest.mark.parametrize("scheme", sorted(CATEGORY))
@pytest.mark.parametrize("steps", [(1,), (3,), (2, 5), (17,)], ids=str)
def test_no_steps_behind_the_last(steps, scheme):
    jobs = [(P.vortex(40 + 15 * k, k), n) for k, n in enumerate(steps)]
    eng = swm.Engine()
    ids = [eng.submit(p, n, timescheme=scheme, hp_association=swm.HP_BY_NODE) for p, n in jobs]
    eng.profile(True)
    while eng.run(16)[0]:
        pass
    eng.profile(False)
    name, per = CATEGORY[scheme]
    assert eng.profile_read()[name][1] == per * max(steps)
    for (p, n), j in zip(jobs, ids):
        o = Oracle(p, scheme, hp_by_node=True)
        for _ in range(n):
            o.step(o.timestep()[0])
        assert same_bits(eng.fetch(j), o.get_U())
