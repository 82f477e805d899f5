"""The midsolve's tiles on the CPU (no GPU): where each tile is stored and read for every number
of empty cells, and whole boards swept by the tables against the oracle, at the sizes around
the tiles' seven low cells (one tile, the first high cells, several steps)."""
import ctypes as C
import os
import subprocess
import tempfile

import numpy as np
import pytest

from oracle import oracle as O
from tests.common import random_sides

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pentago_amd", "csrc")


@pytest.fixture(scope="module")
def mc():
    so = os.path.join(tempfile.mkdtemp(), "midcheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", so,
                           os.path.join(HERE, "hostcheck", "midcheck.cc"), os.path.join(CSRC, "mid_tiles.cc"),
                           os.path.join(CSRC, "mid.cc"), os.path.join(CSRC, "tables.cc")])
    return C.CDLL(so)


@pytest.mark.parametrize("spots", range(19))
def test_tiles_are_stored_until_read(mc, spots):
    assert mc.mc_layout(spots) == 0


@pytest.mark.parametrize("spots", [0, 1, 6, 7, 8, 13, 18])
def test_device_tables(mc, spots):
    assert mc.mc_device_tables(spots) == 0


@pytest.mark.parametrize("stones", [24, 25, 26, 27, 28, 29, 34, 35, 36])
def test_tile_sweep_matches_oracle(mc, stones):
    rng = np.random.default_rng(stones)
    for middle in (0, 1):
        s0, s1 = random_sides(rng, (stones + 1) // 2, stones // 2)
        ply = 2 * stones - middle
        res = np.zeros((19, 4), dtype=np.uint64)
        assert mc.mc_solve(C.c_uint64(s0), C.c_uint64(s1), C.c_uint32(ply), res.ctypes.data_as(C.c_void_p)) == 0
        expect = O.midsolve_internal(O.High((O.C.c_uint64 * 2)(s0, s1), ply))[:37 - stones]
        got = [tuple(int(res[k, 2 * h]) | int(res[k, 2 * h + 1]) << 64 for h in (0, 1)) for k in range(37 - stones)]
        assert got == [tuple(e) for e in expect]
