"""The form for ragged blocks in its other uses: results ORed into the output, partials in more
than two passes, and line plans large enough to be split, against the full blocks' form (plans of
one section, single lines), which other tests check against the oracle."""
import ctypes as C
import random

import numpy as np
import pytest

import pentago_amd as P
from pentago_amd import hip
from tests.test_gpu_ragged_blocks import check, children_of, pick, shape_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("passes", [((0xf, 1),), ((0b0101, 0), (0b1010, 1)), ((0b0001, 2), (0b0110, 4), (0b1000, 3))])
def test_sections_merged_and_in_passes(passes):
    secs = pick(32, 1500000, 4)
    check(secs, children_of(secs), lambda outs, kids: [P.Plan.slab_dims(outs, kids, d, accumulate=a) for d, a in passes])


def ragged_lines(counts):
    """Random lines through a section's last blocks until a plan of them is split."""
    rng = random.Random(7)
    shape = shape_of(counts)
    per = [[min(8, n - 8 * b) for b in range((n + 7) // 8)] for n in shape]
    lines, total = [], 0
    while total < 20000:
        d = rng.choice([a for a in range(4) if sum(counts[a]) < 9])
        base = [rng.randrange(len(per[a])) if rng.random() < 0.3 else len(per[a]) - 1 for a in range(4)]
        for k in range(len(per[d])):
            n = [per[a][k if a == d else base[a]] for a in range(4)]
            w = (n[1] * n[2] * n[3] + 63) // 64
            if 5 * w <= 4 * n[1]:
                total += n[0] * (n[1] - w)
        lines.append(P.make_line(counts, d, tuple(base[a] for a in range(4) if a != d)))
    return lines


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("counts", [((1, 7), (1, 7), (7, 1), (7, 1)), ((5, 4), (1, 7), (7, 1), (2, 3)),
                                    ((4, 5), (5, 4), (1, 7), (7, 2))])
def test_line_plans(counts, accumulate):
    P.init()
    L = P.lib()
    jobs, kept, single = [], [], []
    for k, line in enumerate(ragged_lines(counts)):
        info = P.line_describe(line)
        inp = None
        if info.input_nodes:
            inp = hip.Buffer(64 * info.input_nodes)
            P.fill_seeded(inp.ptr, info.input_nodes, 300 + k)
        out, one = hip.Buffer(64 * info.output_nodes), hip.Buffer(64 * info.output_nodes)
        P.fill_seeded(out.ptr, info.output_nodes, 9000 + k)
        before = out.download(np.zeros(8 * info.output_nodes, dtype=np.uint64))
        jobs.append({"line": line, "input": inp and inp.ptr, "output": out.ptr, "accumulate": accumulate})
        assert L.pe_end_compute_line(C.byref(line), inp and inp.ptr, one.ptr, None) == 0
        kept.append((inp, out, one))
        single.append((out, one, before))
    plan = P.Plan(jobs)
    plan.run()
    hip.synchronize()
    for k, (out, one, before) in enumerate(single):
        got, expect = (m.download(np.zeros_like(before)) for m in (out, one))
        assert np.array_equal(got, expect | before if accumulate else expect), k
    plan.close()
