"""What the tuner leaves in a plan besides its pick."""
import numpy as np
import pytest

from rbsptrsv import SCHED_AUTO, SCHED_BLOCKED, SCHED_FLOW, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [lambda: gen.powerlaw(300_000, seed=3),
                                  lambda: gen.random_lower(20000, 200, seed=2, window=3000)],
                         ids=["powerlaw", "long-rows"])
def test_refinement_on_the_walk_has_its_blocks_timed(make):
    """A mixed plan on the flow schedule refines on the block walk: the same
    blocks are timed as for a plan that only walks."""
    from rbsptrsv import Plan
    f = make().transpose()
    p = Plan.from_factor(f, mixed=True)
    assert p.schedule() == SCHED_FLOW
    q = Plan.from_factor(f, schedule=SCHED_BLOCKED)
    timed = [np.asarray(r.block_kernels()["tuned_ms"]) > 0 for r in (p, q)]
    p.close()
    q.close()
    assert timed[1].any()
    assert np.array_equal(*timed)


@pytest.mark.parametrize("mode,kern", [(2, 1), (3, 2)])
def test_block_kernels_asked_for_are_kept(mode, kern):
    """... also where another schedule is clearly faster than the walk."""
    from rbsptrsv import Plan
    f = gen.banded(20000, seed=4)
    got = []
    for schedule in (SCHED_AUTO, SCHED_BLOCKED):
        p = Plan.from_factor(f, schedule=schedule, block_kernels=mode)
        got.append(p.block_kernels()["kern"])
        p.close()
    assert kern in got[1]
    assert np.array_equal(*got)
