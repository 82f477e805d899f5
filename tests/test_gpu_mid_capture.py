"""Runs of a batched plan captured into a caller's graph: its replays, what becomes of the plan's
memory, and the launches that a plan reports."""
import numpy as np
import pytest

import pentago_amd as P
from pentago_amd.workloads import seeded_board, seeded_boards
from tests.graph_capture import Captured

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    P.init()


def boards_of(stones, seed=5):
    rng = np.random.default_rng(seed)
    return [seeded_board(rng, s) for s in stones]


@pytest.mark.parametrize("streams", [-1, 2])
def test_captured_run_and_closed_plan(streams):
    """Replays equal eager runs; the memory of a plan that was captured is not handed on, since a
    replay of the caller's may still use it."""
    P.release_kept_memory()
    boards = seeded_boards(40, 61, 20, 32)
    expect = P.midsolve_batch(boards, mode=0)
    plan = P.MidPlan(boards, streams=streams, use_graph=False)
    graph = Captured(plan.run)
    for _ in range(3):
        graph.replay()
        assert P.results_to_lists(boards, plan.results(graph.stream.ptr)) == expect
        plan.run()
        assert P.results_to_lists(boards, plan.results()) == expect
    graph.close()
    plan.close()
    assert P.kept_memory_bytes() == 0


@pytest.mark.parametrize("threads", [256, 512, 1024, 0])
def test_threads_asked_for_are_run_and_reported(threads):
    """Few boards of several tiles: the size that a plan without one asked for would change."""
    boards = boards_of([26] * 3 + [30] * 4)
    plan = P.MidPlan(boards, threads=threads, use_graph=False)
    graph = Captured(plan.run)
    info, blocks = plan.info(), sorted(b for _, b in graph.kernels())
    graph.close()
    assert info["large_boards"] == 0
    assert blocks == sorted([1, 256, info["threads"]])     # queue head, tables, boards
    if threads:
        assert info["threads"] == threads
    plan.run()
    got = P.results_to_lists(boards, plan.results())
    plan.close()
    assert got == P.midsolve_batch(boards, mode=0)


@pytest.mark.parametrize("stones", [[18], [19, 20, 21, 28, 29], [22, 35]])
def test_launches_reported_are_launched(stones):
    boards = boards_of(stones)
    plan = P.MidPlan(boards, small_spots=8, use_graph=False)
    graph = Captured(plan.run)
    launched = len(graph.kernels())
    graph.close()
    assert plan.info()["launches"] == launched
    assert P.mid_schedule_info(boards, int(200e9), small_spots=8)[0] >= launched
    plan.close()
