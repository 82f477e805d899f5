"""The queue-fed launch form on plans of few blocks (fewer than XCDs, one more, one less, odd
numbers) against the static grid."""
import numpy as np
import pytest

import pentago_amd as P
from pentago_amd import hip

pytestmark = pytest.mark.gpu

BLOCK = 4096
COUNTS = ((3, 4), (4, 4), (4, 4), (4, 3))


@pytest.mark.parametrize("box", [(1, 1, 1, 1), (1, 1, 1, 7), (1, 2, 2, 2), (1, 3, 3, 1), (17, 1, 1, 1), (2, 2, 2, 3)])
def test_queue_equals_grid(box):
    P.init()
    nb = [(s + 7) // 8 for s in P.section_shape(COUNTS)]
    lo = [n - b for n, b in zip(nb, box)]      # the section's last blocks
    kids, kept = [], []
    for d in range(4):
        info = P.line_describe(P.make_line(COUNTS, d, tuple(lo[a] for a in range(4) if a != d)))
        child, perm = info.standard_child.counts, list(info.permutation)
        n = [(s + 7) // 8 for s in P.section_shape(child)]
        clo = [0 if c == info.child_dimension else lo[perm[c]] for c in range(4)]
        chi = [n[c] if c == info.child_dimension else nb[perm[c]] for c in range(4)]
        nodes = BLOCK * int(np.prod([h - l for l, h in zip(clo, chi)]))
        m = hip.Buffer(64 * nodes)
        P.fill_seeded(m.ptr, nodes, 40 + d)
        kept.append(m)
        kids.append(P.Slab.of(child, clo, chi, m.ptr))
    nodes = BLOCK * int(np.prod(box))
    out = hip.Buffer(64 * nodes)
    plan = P.Plan.slab(P.Slab.of(COUNTS, lo, nb, out.ptr), kids)
    expect = None
    for form in (0, 1, 6):
        P.fill_seeded(out.ptr, nodes, 7)
        plan.set_launch(form)
        plan.run()
        hip.synchronize()
        got = out.download(np.zeros(8 * nodes, dtype=np.uint64))
        if expect is None:
            expect = got
        assert np.array_equal(got, expect), form
    plan.close()
