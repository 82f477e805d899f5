"""The midsolve's tile records made a piece at a time, as they are uploaded (no GPU): pieces that end
inside a number of empty cells, at its end and past the last tile."""
import ctypes as C
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pentago_amd", "csrc")


@pytest.fixture(scope="module")
def rc():
    so = os.path.join(tempfile.mkdtemp(), "recordcheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", so,
                           os.path.join(HERE, "hostcheck", "recordcheck.cc"), os.path.join(CSRC, "mid_tiles.cc"),
                           os.path.join(CSRC, "mid.cc"), os.path.join(CSRC, "tables.cc")])
    return C.CDLL(so)


@pytest.mark.parametrize("piece", [1000, 8192, 59049, 1 << 20])
def test_pieces_equal_the_whole(rc, piece):
    assert rc.rc_pieces(C.c_int64(piece)) == 0
