"""Plans on both sides of the rule for a small board's workgroup (few largest boards, more of them
than compute units, boards of a single tile) against plans with 256 threads."""
import numpy as np
import pytest

import pentago_amd as P
from pentago_amd.workloads import seeded_board

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stones", [[28] * 300, [23] + [28, 27, 29] * 13, [29] * 40, [26, 34] * 20, [22]])
def test_plans_agree(stones):
    P.init()
    rng = np.random.default_rng(len(stones))
    boards = [seeded_board(rng, s) for s in stones]
    got = []
    for threads in (0, 256):
        plan = P.MidPlan(boards, threads=threads)
        plan.run()
        got.append(plan.results())
        plan.close()
    assert np.array_equal(got[0], got[1])
