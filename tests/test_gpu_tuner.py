"""What the tuner leaves in a plan besides its pick."""
import numpy as np
import pytest

from rbsptrsv import SCHED_AUTO, SCHED_BLOCKED, SCHED_FLOW, SCHED_LEVEL, gen

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


def test_losing_schedules_leave_nothing():
    """A plan holds the tables of the schedule it runs, as if asked for by
    name, not those of the others that were built and timed."""
    from rbsptrsv import Plan
    f = gen.banded(20000, seed=4).transpose()
    held = []
    for schedule in (SCHED_AUTO, SCHED_LEVEL):
        # (for many columns the fused schedule is built besides)
        p = Plan.from_factor(f, schedule=schedule, tune_rhs=32)
        assert p.schedule() == SCHED_LEVEL
        held.append(p.info().device_bytes)
        p.close()
    assert held[0] == held[1]
