"""Memory that a closed plan leaves to the next one, as its caller sees it: budgets that default to
the free memory, and a call that gives it back."""
import pytest

import pentago_amd as P
from pentago_amd import hip
from pentago_amd.workloads import seeded_boards

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    P.init()


def solve(boards, **kw):
    """A plan's whole life; its info() and answers."""
    plan = P.MidPlan(boards, **kw)
    info = plan.info()
    plan.run()
    got = P.results_to_lists(boards, plan.results())
    plan.close()
    return info, got


def test_default_budget_after_a_closed_plan():
    """The kept block is memory that the next plan may have: its default budget is the same."""
    solve(seeded_boards(4, 3, 28, 30))      # first use of the kernels, small block
    boards = seeded_boards(100, 90, 22, 22)
    first, expect = solve(boards)
    kept = first["workspace_bytes"]
    assert kept > 1 << 30
    second, got = solve(boards)
    assert got == expect
    assert second["workgroups"] == first["workgroups"]
    # 60 % of the free memory, which the kept block must not take part of away
    assert second["workspace_budget"] > first["workspace_budget"] - 0.1 * kept


def test_kept_memory_can_be_released():
    boards = seeded_boards(100, 90, 22, 22)
    solve(boards)
    kept = P.kept_memory_bytes()
    assert kept > 1 << 30
    free = hip.mem_info()[0]
    P.release_kept_memory()
    assert P.kept_memory_bytes() == 0
    # freed or not: the driver's own count moves by a few MB beside it
    assert hip.mem_info()[0] - free > kept // 2
    P.release_kept_memory()      # nothing kept: nothing to do
    _, got = solve(boards[:3])
    assert got == P.midsolve_batch(boards[:3], mode=0)


def test_a_plan_reports_the_memory_that_it_holds():
    """A plan in the kept block of a larger one holds that block, unless its budget is smaller."""
    P.release_kept_memory()
    large, small = seeded_boards(100, 90, 22, 22), seeded_boards(70, 91, 22, 22)
    need = P.mid_schedule_info(small, int(200e9), workgroups=512, threads=512, streams=2)[1]
    held = solve(large)[0]["workspace_bytes"]
    assert need < held < 2 * need and P.kept_memory_bytes() == held
    info, got = solve(small)
    assert info["workspace_bytes"] == held
    assert got == P.midsolve_batch(small, mode=0)
    info, got = solve(small, workspace_budget=need)
    assert info["workspace_bytes"] == need
    assert got == P.midsolve_batch(small, mode=0)


def test_a_plan_and_the_kept_block_within_the_budget():
    P.release_kept_memory()
    small = seeded_boards(40, 92, 22, 22)
    need = P.mid_schedule_info(small, int(200e9), workgroups=512, threads=512, streams=2)[1]
    solve(seeded_boards(100, 90, 22, 22))
    kept = P.kept_memory_bytes()
    assert kept > 2 * need
    plan = P.MidPlan(small, workspace_budget=kept + 2 * need)    # room for both
    assert P.kept_memory_bytes() == kept
    plan.close()
    assert P.kept_memory_bytes() == kept                         # the larger block stays
    plan = P.MidPlan(small, workspace_budget=kept)               # room for the kept block or the plan
    assert plan.info()["workspace_bytes"] <= kept and P.kept_memory_bytes() == 0
    plan.run()
    assert P.results_to_lists(small, plan.results()) == P.midsolve_batch(small, mode=0)
    plan.close()


def test_the_larger_block_is_kept_while_it_is_used():
    P.release_kept_memory()
    large, small = seeded_boards(100, 90, 22, 22), seeded_boards(40, 92, 22, 22)
    held = solve(large)[0]["workspace_bytes"]
    for _ in range(3):                                           # in turn
        own = solve(small)[0]["workspace_bytes"]
        assert own < held // 2 and P.kept_memory_bytes() == held
        assert solve(large)[0]["workspace_bytes"] == held
    solve(small)
    solve(small)                                                 # no large plan any more
    assert P.kept_memory_bytes() == own
