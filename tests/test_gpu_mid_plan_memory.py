"""Plans made, run and closed in a row take over the memory of the one before (sizes that fit,
larger and smaller ones), also from several threads: every answer equals the plain solve."""
import threading

import pytest

import pentago_amd as P
from pentago_amd.workloads import seeded_boards

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    P.init()


def solve(boards, **kw):
    plan = P.MidPlan(boards, **kw)
    plan.run()
    got = P.results_to_lists(boards, plan.results())
    plan.close()
    return got


@pytest.mark.parametrize("sizes", [(24, 24, 20, 40, 3, 24), (1, 60, 59, 61, 1)])
def test_plans_in_a_row(sizes):
    for k, n in enumerate(sizes):
        boards = seeded_boards(n, 50 + k, 22, 30)
        assert solve(boards) == P.midsolve_batch(boards, mode=0), (k, n)


def test_plans_of_several_threads():
    batches = [seeded_boards(16 + k, 80 + k, 23, 30) for k in range(4)]
    expect = [P.midsolve_batch(b, mode=0) for b in batches]
    wrong = []

    def work(k):
        for _ in range(6):
            if solve(batches[k]) != expect[k]:
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_plan_within_its_budget():
    """A plan whose budget is below the kept block's size gets memory of its own."""
    large, small = seeded_boards(80, 90, 22, 24), seeded_boards(40, 91, 22, 24)
    expect = P.midsolve_batch(small, mode=0)
    solve(large)
    plan = P.MidPlan(small)
    need = plan.info()["workspace_bytes"]
    plan.close()
    solve(large)
    plan = P.MidPlan(small, workspace_budget=need)
    assert plan.info()["workspace_bytes"] <= need
    plan.run()
    assert P.results_to_lists(small, plan.results()) == expect
    plan.close()
