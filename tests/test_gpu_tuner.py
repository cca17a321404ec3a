"""What the tuner leaves in a plan besides its pick."""
import numpy as np
import pytest

from rbsptrsv import SCHED_BLOCKED, SCHED_FLOW, gen

pytestmark = pytest.mark.gpu


def test_refinement_on_the_walk_has_its_blocks_timed():
    """A mixed plan on the flow schedule refines on the block walk: the same
    blocks are timed as for a plan that only walks."""
    from rbsptrsv import Plan
    f = gen.powerlaw(300_000, seed=3).transpose()
    p = Plan.from_factor(f, lv=3, mixed=True)
    assert p.schedule() == SCHED_FLOW
    q = Plan.from_factor(f, lv=3, schedule=SCHED_BLOCKED)
    timed = [np.asarray(r.block_kernels()["tuned_ms"]) > 0 for r in (p, q)]
    p.close()
    q.close()
    assert timed[1].sum() > 4
    assert np.array_equal(*timed)
