"""Work that programs built on this engine have it do, as cases that can be timed.

The engine has two halves.  The end engine computes superscore nodes (64 bytes each: we-win,
we-win-or-tie) of sections of the game from the nodes of their child sections: single block
lines as a slice loop schedules them, boxes of blocks, whole slices, sections run in passes.
The midsolve solves one position (18 or more stones) by a sweep over everything below it: one
board for a player, batches of boards for an analysis, a request stream for a server.  The
cases below cover both from the smallest call to the largest, with the section shapes, stone
counts and options of the repository's own benchmark and tests.

Every output is exact bits (no rounding anywhere), so results of two builds are compared for
equality.
"""
import ctypes as C
import random

import numpy as np
import torch

import pentago_amd as P
from pentago_amd.workloads import seeded_board

BLOCK = 4096   # node slots per 8x8x8x8 block of a slab

# Sections by name: per-quadrant (black, white) stone counts, standard form.
SECTIONS = {
    "24-33333333": ((3, 3), (3, 3), (3, 3), (3, 3)),   # the benchmark's headline section, 420^4
    "24-33243342": ((3, 3), (2, 4), (3, 3), (4, 2)),   # mixed with it in the same launch
    "30-34444443": ((3, 4), (4, 4), (4, 4), (4, 3)),   # slice 30: reflected children, 318x160x160x318
    "31-35265362": ((3, 5), (2, 6), (5, 3), (6, 2)),   # shallow quadrants, every shape ragged
    "32-17177171": ((1, 7), (1, 7), (7, 1), (7, 1)),   # 18 nodes a side
    "29-54177123": ((5, 4), (1, 7), (7, 1), (2, 3)),   # quadrant 0 full: three open dimensions
}


class DeviceMemory:
    """Device memory as the engine takes it (an address and a size), backed by a tensor."""

    def __init__(self, words):
        self.tensor = torch.zeros(int(words), dtype=torch.int64, device="cuda")
        self.ptr = self.tensor.data_ptr()
        self.nbytes = 8 * self.tensor.numel()


def seeded_memory(nodes, seed):
    m = DeviceMemory(8 * nodes)
    P.fill_seeded(m.ptr, int(nodes), int(seed))
    return m


def blocks_of(lo, hi):
    return int(np.prod([h - l for l, h in zip(lo, hi)]))


def nodes_in(shape, lo, hi):
    return int(np.prod([min(s, 8 * h) - 8 * l for s, l, h in zip(shape, lo, hi)]))


def open_dims(counts):
    return [d for d in range(4) if sum(counts[d]) < 9]


def child_box(counts, d, lo, hi):
    """The child section, its block box and the child nodes that dimension d's lines through
    the box [lo, hi) read."""
    info = P.line_describe(P.make_line(counts, d, tuple(lo[a] for a in range(4) if a != d)))
    child, cd, perm = info.standard_child.counts, info.child_dimension, list(info.permutation)
    cshape = P.section_shape(child)
    clo = tuple(0 if c == cd else lo[perm[c]] for c in range(4))
    chi = tuple((cshape[c] + 7) // 8 if c == cd else hi[perm[c]] for c in range(4))
    return child, clo, chi, nodes_in(cshape, clo, chi)


# ---- the ranges ----

def box_of(name, at, side):
    """A box of at most side^4 blocks of a section, from block `at` (or as near as it fits), so
    that boxes that reach the section's end hold its partial blocks."""
    nb = [(s + 7) // 8 for s in P.section_shape(SECTIONS[name])]
    lo = [max(0, min(at, n - side)) for n in nb]
    return lo, [min(n, l + side) for n, l in zip(nb, lo)]


def listed():
    return [
        # One block line, the unit that a slice loop hands out, of a small ragged section: the
        # smallest call of the end engine, where the launch itself counts.
        {"name": "line", "kind": "lines", "section": "32-17177171", "lines": 1, "wakeup": False},
        # A slice loop's burst: whole lines of the headline section in all four dimensions, one
        # asynchronous call and one wakeup each.
        {"name": "lines", "kind": "lines", "section": "24-33333333", "lines": 48, "wakeup": True},
        # A box of blocks at the ragged end of a section whose children are reflected, from a
        # kept plan: an ordinary share of work.
        {"name": "box_ragged", "kind": "box", "section": "30-34444443", "at": 99, "side": 5, "second": "", "second_side": 0},
        # The benchmark's headline launch at a size that leaves room for other work on the card:
        # two sections of slice 24 in one plan.
        {"name": "box_large", "kind": "box", "section": "24-33333333", "at": 4, "side": 14, "second": "24-33243342", "second_side": 6},
        # A section too large to hold with all its children runs in passes over subsets of its
        # dimensions: children of dimensions 1-3 into a partial, then dimension 0 finishes it.
        {"name": "passes", "kind": "passes", "section": "30-34444443", "at": 0, "side": 10, "first": 0b1110},
        # A group of a slice's sections computed from the next slice's store and counted, plans
        # built on the way: the step of the slice driver.
        {"name": "slice_group", "kind": "slice", "slice": 34, "sections": 96, "skip": 540},
        # Blocks of a file brought into a slab, counted, and turned back into file words.
        {"name": "file_blocks", "kind": "file", "section": "31-35265362", "at": 0, "side": 11, "filter": 1},
        # One position of an ongoing game near its end: a player waits for it.
        {"name": "mid_one", "kind": "mid_one", "stones": 26},
        # The deepest position the solver takes.
        {"name": "mid_deep", "kind": "mid_one", "stones": 18},
        # A batch of late positions, each batch new: plan, run and results.
        {"name": "mid_late", "kind": "mid_batch", "boards": 2048, "least": 24, "most": 30, "kept": False},
        # The benchmark's mix of 18 to 30 stones in a kept plan.
        {"name": "mid_mix", "kind": "mid_batch", "boards": 65, "least": 18, "most": 30, "kept": True},
        # Requests to the serving loop, all submitted at once and waited for.
        {"name": "serve", "kind": "serve", "requests": 96, "least": 18, "most": 34},
    ]


def log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["lines", "box", "box", "passes", "slice", "file", "mid_one", "mid_batch", "mid_batch", "serve"])
    if kind == "lines":
        return {"kind": kind, "section": rng.choice(sorted(SECTIONS)), "lines": log_int(rng, 1, 48),
                "wakeup": rng.random() < 0.5}
    if kind == "box":
        case = {"kind": kind, "section": rng.choice(sorted(SECTIONS)), "at": rng.randrange(0, 50),
                "side": log_int(rng, 1, 12), "second": "", "second_side": 0}
        if rng.random() < 0.4:   # sections of one plan may have any stone count up to 34
            case["second"] = rng.choice(sorted(set(SECTIONS) - {case["section"]}))
            case["second_side"] = log_int(rng, 1, 6)
        return case
    if kind == "passes":
        name = rng.choice(["24-33333333", "30-34444443", "31-35265362", "32-17177171"])
        return {"kind": kind, "section": name, "at": rng.randrange(0, 40), "side": log_int(rng, 2, 10),
                "first": rng.choice([0b1110, 0b0111, 0b1100, 0b0011, 0b1010, 0b1000])}
    if kind == "slice":
        return {"kind": kind, "slice": rng.choice([33, 34, 34, 35]), "sections": log_int(rng, 4, 60),
                "skip": rng.randrange(100, 240)}
    if kind == "file":
        return {"kind": kind, "section": rng.choice(sorted(SECTIONS)), "at": rng.randrange(0, 40),
                "side": log_int(rng, 1, 11), "filter": rng.choice([0, 1, 1])}
    if kind == "mid_one":
        return {"kind": kind, "stones": rng.randint(18, 35)}
    if kind == "mid_batch":
        least = rng.randint(18, 30)
        most = min(34, least + rng.randint(0, 10))
        return {"kind": kind, "boards": log_int(rng, 4, {18: 48, 19: 64, 20: 128, 21: 256, 22: 512}.get(least, 2048)),
                "least": least, "most": most, "kept": rng.random() < 0.5}
    least = rng.randint(18, 26)
    return {"kind": "serve", "requests": log_int(rng, 2, 96), "least": least, "most": min(34, least + rng.randint(4, 16))}


# ---- the inputs ----

def line_list(case):
    """The case's lines: dimensions in turn, block bases spread over the section, the last
    (partial) blocks among them."""
    counts = SECTIONS[case["section"]]
    nb = [(s + 7) // 8 for s in P.section_shape(counts)]
    rng = random.Random(case["lines"])
    dims = open_dims(counts)
    out = []
    for k in range(case["lines"]):
        d = dims[k % len(dims)]
        base = tuple(nb[a] - 1 if k % 5 == 4 else rng.randrange(nb[a]) for a in range(4) if a != d)
        out.append(P.make_line(counts, d, base))
    return out


def boxes(case):
    got = [(case["section"],) + tuple(map(tuple, box_of(case["section"], case["at"], case["side"])))]
    if case.get("second"):
        got.append((case["second"],) + tuple(map(tuple, box_of(case["second"], case["at"], case["second_side"]))))
    return got


def box_children(specs):
    """The child boxes (child section, lo, hi) that the boxes' lines read, each once however many
    dimensions read it, and their nodes."""
    keys, nodes = [], 0
    for name, lo, hi in specs:
        counts = SECTIONS[name]
        for d in open_dims(counts):
            child, clo, chi, n = child_box(counts, d, lo, hi)
            if (child, clo, chi) not in keys:
                keys.append((child, clo, chi))
                nodes += n
    return keys, nodes


def box_outputs(specs):
    return sum(nodes_in(P.section_shape(SECTIONS[n]), lo, hi) for n, lo, hi in specs)


def make_children(keys, seed):
    slabs, kept = [], []
    for k, (child, lo, hi) in enumerate(keys):
        m = seeded_memory(BLOCK * blocks_of(lo, hi), 1000003 * seed + k)
        kept.append(m)
        slabs.append(P.Slab.of(child, lo, hi, m.ptr))
    return slabs, kept


def slice_sections(case):
    """A run of a slice's sections, from the smallest on (skip: where the run begins)."""
    secs = P.descendent_sections(((0, 0),) * 4, case["slice"])
    secs = sorted(secs, key=lambda s: (int(np.prod(P.section_shape(s))), P.section_sig(s)))
    at = min(case["skip"], len(secs) - case["sections"])
    return secs[at:at + case["sections"]]


def children_of(secs):
    turn = sum(map(sum, secs[0])) & 1
    out = set()
    for s in secs:
        for q in open_dims(s):
            c = [list(x) for x in s]
            c[q][turn] += 1
            out.add(P.standardize(tuple(map(tuple, c)))[0])
    return sorted(out)


def stone_counts(n, least, most):
    """Stone counts of n boards, every count of the range in turn."""
    return [least + k % (most - least + 1) for k in range(n)]


def make_boards(stones, seed):
    rng = np.random.default_rng(seed)
    return [seeded_board(rng, s) for s in stones]


def prepare(case, seed):
    P.init()
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "lines":
        s["jobs"], s["out"], s["kept"], s["wakeup"] = [], [], [], case["wakeup"]
        for k, line in enumerate(line_list(case)):
            info = P.line_describe(line)
            inp = seeded_memory(info.input_nodes, 1000003 * seed + k)
            out = DeviceMemory(8 * info.output_nodes)
            s["jobs"].append((line, inp.ptr, out.ptr))
            s["out"].append(out.tensor)
            s["kept"].append(inp)
    elif kind in ("box", "passes"):
        specs = boxes(case)
        keys, _ = box_children(specs)
        kids, s["kept"] = make_children(keys, seed)
        mem = [DeviceMemory(8 * BLOCK * blocks_of(lo, hi)) for _, lo, hi in specs]
        outs = [P.Slab.of(SECTIONS[n], lo, hi, m.ptr) for (n, lo, hi), m in zip(specs, mem)]
        s["out"] = [m.tensor for m in mem]
        if kind == "box":
            s["plans"] = [P.Plan.slab(outs, kids)]
        else:
            s["plans"] = [P.Plan.slab_dims(outs, kids, case["first"], accumulate=2),
                          P.Plan.slab_dims(outs, kids, 0xf & ~case["first"], accumulate=3)]
    elif kind == "slice":
        secs = slice_sections(case)
        random.Random(seed).shuffle(secs)   # a driver takes its sections in any order
        s["arena"] = DeviceMemory(P.slice_bytes(secs) // 8)
        s["store"] = P.SliceStore(secs, arena=s["arena"])
        s["children"] = None
        if case["slice"] < 35:
            kids = children_of(secs)
            s["kids_arena"] = seeded_memory(P.slice_bytes(kids) // 64, seed)
            s["children"] = P.SliceStore(kids, arena=s["kids_arena"])
    elif kind == "file":
        (name, lo, hi), = boxes(dict(case, second=""))
        n = BLOCK * blocks_of(lo, hi)
        s["nodes"], s["filter"], s["turn"] = n, case["filter"], sum(map(sum, SECTIONS[name])) & 1
        s["words"] = seeded_memory(n, seed)   # a file's blocks, decompressed
        s["slab_mem"], s["back"] = DeviceMemory(8 * n), DeviceMemory(8 * n)
        s["slab"] = P.Slab.of(SECTIONS[name], lo, hi, s["slab_mem"].ptr)
        s["counts"] = DeviceMemory(4 * s["slab"].blocks)
    elif kind == "mid_one":
        s["board"], = make_boards([case["stones"]], seed)
    elif kind == "mid_batch":
        s["boards"] = make_boards(stone_counts(case["boards"], case["least"], case["most"]), seed)
        s["plan"] = P.MidPlan(s["boards"]) if case["kept"] else None
    else:
        s["boards"] = make_boards(stone_counts(case["requests"], case["least"], case["most"]), seed)
        s["server"] = P.MidServer()
    return s


# ---- a pass ----

def run_server(s):
    """Submit every board, then take each answer (the C entry points, as a server process
    calls them)."""
    L, server = P.lib(), s["server"].ptr
    out = np.zeros((len(s["boards"]), 19, 4), dtype=np.int64)
    tickets = (C.c_int64 * len(s["boards"]))()
    latency = C.c_double()
    for k, b in enumerate(s["boards"]):
        st = L.pe_mid_server_submit(server, C.byref(b), C.cast(C.byref(tickets, 8 * k), C.POINTER(C.c_int64)))
        if st:
            raise P.PentagoError(L.pe_last_error().decode())
    for k in range(len(s["boards"])):
        if L.pe_mid_server_wait(server, tickets[k], out[k].ctypes.data, C.byref(latency)):
            raise P.PentagoError(L.pe_last_error().decode())
    return out


@P.WAKEUP
def woken(ctx):
    """A line's completion callback, called on a runtime thread (one object that outlives every
    call)."""


def run(state):
    s, kind = state, state["kind"]
    if kind == "lines":
        L = P.lib()
        for line, i, o in s["jobs"]:
            if s["wakeup"]:
                st = L.pe_end_schedule_line(C.byref(line), i, o, None, woken, None)
            else:
                st = L.pe_end_compute_line(C.byref(line), i, o, None)
            P._check(st, "pe_end_schedule_line")
        return s["out"]
    if kind in ("box", "passes"):
        for plan in s["plans"]:
            plan.run()
        return s["out"]
    if kind == "slice":
        s["store"].compute(s["children"])
        return {"nodes": s["arena"].tensor, "counts": s["store"].counts().view(np.int64)}
    if kind == "file":
        L = P.lib()
        P._check(L.pe_supertensor_decode(s["filter"], s["turn"], s["words"].ptr, s["nodes"], s["slab_mem"].ptr, None),
                 "pe_supertensor_decode")
        P.count_blocks(s["slab"], s["counts"].ptr)
        P._check(L.pe_supertensor_encode(s["filter"], s["turn"], s["slab_mem"].ptr, s["nodes"], s["back"].ptr, None),
                 "pe_supertensor_encode")
        return {"slab": s["slab_mem"].tensor, "counts": s["counts"].tensor, "words": s["back"].tensor}
    if kind == "mid_one":
        out = np.zeros((19, 4), dtype=np.uint64)
        P.midsolve_internal_raw(s["board"], out)
        return out.view(np.int64)
    if kind == "mid_batch":
        plan = s["plan"] or P.MidPlan(s["boards"])
        plan.run()
        out = plan.results().view(np.int64)
        if s["plan"] is None:
            plan.close()
        return out
    return run_server(s)


# ---- what a pass cannot do without ----

def choose(n, k):
    r = 1
    for i in range(k):
        r = r * (n - i) // (i + 1)
    return r


def mid_work(stones):
    """Solving a board: the board in, 19 results out, and for every position of every level
    the OR of its children's 256 bits and the combination with the two sides' wins and their
    rotations (counted as 32-bit logic operations: 8 a child, 100 a position)."""
    spots = 36 - stones
    ops = 0
    for n in range(spots + 1):
        ops += choose(spots, n) * choose(n, n // 2) * (8 * (spots - n) + 100)
    return {"bytes": 24 + 19 * 32, "flops": ops}


def work(case):
    kind = case["kind"]
    if kind == "lines":
        n = sum(i.input_nodes + i.output_nodes for i in map(P.line_describe, line_list(case)))
        return {"bytes": 64 * n, "flops": 0}
    if kind in ("box", "passes"):
        specs = boxes(case)
        return {"bytes": 64 * (box_outputs(specs) + box_children(specs)[1]), "flops": 0}
    if kind == "slice":
        secs = slice_sections(case)
        n = sum(int(np.prod(P.section_shape(s))) for s in secs)
        kids = children_of(secs) if case["slice"] < 35 else []
        # the nodes written, then read once more to count them
        return {"bytes": 64 * (2 * n + sum(int(np.prod(P.section_shape(c))) for c in kids)), "flops": 0}
    if kind == "file":
        (name, lo, hi), = boxes(dict(case, second=""))
        n = nodes_in(P.section_shape(SECTIONS[name]), lo, hi)
        # words in, nodes out, nodes counted, nodes in, words out
        return {"bytes": 64 * 4 * BLOCK * blocks_of(lo, hi) + 64 * n + 32 * blocks_of(lo, hi), "flops": 0}
    if kind == "mid_one":
        return mid_work(case["stones"])
    n = case["boards"] if kind == "mid_batch" else case["requests"]
    got = [mid_work(x) for x in stone_counts(n, case["least"], case["most"])]
    return {"bytes": sum(g["bytes"] for g in got), "flops": sum(g["flops"] for g in got)}
