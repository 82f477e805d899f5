"""Plans whose ragged blocks are launched apart (waves filled in stored order) against plans of one
section each, which keep the form that test_gpu_box.py and test_gpu_section_passes.py check
against the oracle: whole sections of slices 34 and 35 with blocks of every remainder, in one pass
and in passes over subsets of the dimensions."""
import random

import numpy as np
import pytest

import pentago_amd as P
from pentago_amd import hip

pytestmark = pytest.mark.gpu

BLOCK = 4096


def shape_of(s):
    return [int(x) for x in P.section_shape(s)]


def saved_waves(s):
    """Waves that the ragged form saves on the section's blocks that take it."""
    per = [[min(8, n - 8 * b) for b in range((n + 7) // 8)] for n in shape_of(s)]
    total = 0
    for n1 in per[1]:
        for n2 in per[2]:
            for n3 in per[3]:
                w = (n1 * n2 * n3 + 63) // 64
                if 5 * w <= 4 * n1:
                    total += sum(per[0]) * (n1 - w)
    return total


def pick(slice_, largest, open_dims=0):
    """Sections of a slice, in a seeded order, until the plan's ragged blocks are launched apart;
    none larger than `largest` nodes, none that is launched so on its own."""
    secs = [s for s in P.descendent_sections(((0, 0),) * 4, slice_)
            if np.prod(shape_of(s)) <= largest and 0 < saved_waves(s) < 4000 and sum(sum(q) < 9 for q in s) >= open_dims]
    random.Random(slice_).shuffle(secs)
    out, total = [], 0
    for s in secs:
        if total >= 20000:
            break
        out.append(s)
        total += saved_waves(s)
    assert total >= 20000
    return out


def children_of(secs):
    turn = sum(map(sum, secs[0])) & 1
    out = set()
    for s in secs:
        for q in range(4):
            if sum(s[q]) < 9:
                c = [list(x) for x in s]
                c[q][turn] += 1
                out.add(P.standardize(tuple(map(tuple, c)))[0])
    return sorted(out)


class Slabs:
    def __init__(self, secs, seed):
        self.mem, self.slabs = [], []
        for k, s in enumerate(secs):
            nb = [(n + 7) // 8 for n in shape_of(s)]
            nodes = BLOCK * int(np.prod(nb))
            m = hip.Buffer(64 * nodes)
            P.fill_seeded(m.ptr, nodes, seed + k)
            self.mem.append(m)
            self.slabs.append(P.Slab.of(s, (0,) * 4, tuple(nb), m.ptr))


def check(secs, kids, plans):
    """plans: of (output slabs, child slabs), the plans to run in order."""
    P.init()
    child = Slabs(kids, 77)
    together, alone = Slabs(secs, 5), Slabs(secs, 5)
    for plan in plans(together.slabs, child.slabs):
        plan.run()
    for slab in alone.slabs:
        for plan in plans([slab], child.slabs):
            plan.run()
    hip.synchronize()
    for s, a, b in zip(secs, together.mem, alone.mem):
        x, y = (m.download(np.zeros(m.nbytes // 8, dtype=np.uint64)) for m in (a, b))
        assert np.array_equal(x, y), s


@pytest.mark.parametrize("slice_,largest", [(34, 400000), (34, 4000000), (35, 600000)])
def test_whole_sections(slice_, largest):
    secs = pick(slice_, largest)
    check(secs, children_of(secs) if slice_ < 35 else [], lambda outs, kids: [P.Plan.slab(outs, kids)])


@pytest.mark.parametrize("first", [0b0011, 0b0101, 0b1110])
def test_passes(first):
    secs = pick(32, 1500000, 4)
    check(secs, children_of(secs),
          lambda outs, kids: [P.Plan.slab_dims(outs, kids, first, accumulate=2),
                              P.Plan.slab_dims(outs, kids, 0xf & ~first, accumulate=3)])
