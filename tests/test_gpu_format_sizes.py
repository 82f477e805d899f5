"""Decode and encode of supertensor words at the kernel's edges (one node, part of a quad's wave, of a
workgroup, the first size past the caches), against the definition of the interleave filter on
bits, apart and in place."""
import numpy as np
import pytest

import pentago_amd as P
from pentago_amd import hip

pytestmark = pytest.mark.gpu


def reference(words, filter_, turn):
    """(we-win, we-win-or-tie) of file words, node by node on bits."""
    bits = np.unpackbits(words.view(np.uint8).reshape(-1, 64), axis=1, bitorder="little")
    if filter_:
        black, white = bits[:, 0::2], bits[:, 1::2]
    else:
        black, white = bits[:, :256], bits[:, 256:]
    out = np.concatenate([white, 1 - black], axis=1) if turn else np.concatenate([black, 1 - white], axis=1)
    return np.packbits(out, axis=1, bitorder="little").view(np.uint64).reshape(-1, 8)


@pytest.mark.parametrize("filter_,turn", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("nodes", [1, 3, 15, 63, 64, 65, 255, 256, 257, 4099, (1 << 21) + 5])
def test_sizes(nodes, filter_, turn):
    P.init()
    rng = np.random.default_rng(nodes)
    words = rng.integers(0, 1 << 64, size=(nodes, 8), dtype=np.uint64)
    at = np.unique(np.concatenate([np.arange(min(nodes, 300)), np.arange(max(0, nodes - 300), nodes)]))
    guard = np.full(8, 0x5A5A5A5A5A5A5A5A, dtype=np.uint64)   # nothing is written past the last node
    src, dst = hip.Buffer(64 * nodes + 64), hip.Buffer(64 * nodes + 64)
    src.upload(words)
    src.upload(guard, 64 * nodes)
    dst.upload(guard, 64 * nodes)
    run = P.lib().pe_supertensor_decode, P.lib().pe_supertensor_encode

    def down(b):
        hip.synchronize()
        a = b.download(np.zeros(8 * nodes + 8, dtype=np.uint64))
        assert np.array_equal(a[8 * nodes:], guard)
        return a[:8 * nodes].reshape(-1, 8)

    P._check(run[0](filter_, turn, src.ptr, nodes, dst.ptr, None), "decode")
    got = down(dst)
    assert np.array_equal(got[at], reference(words[at], filter_, turn))
    P._check(run[0](filter_, turn, src.ptr, nodes, src.ptr, None), "decode in place")
    assert np.array_equal(down(src), got)
    P._check(run[1](filter_, turn, dst.ptr, nodes, src.ptr, None), "encode")
    assert np.array_equal(down(src), words)
    P._check(run[1](filter_, turn, dst.ptr, nodes, dst.ptr, None), "encode in place")
    assert np.array_equal(down(dst), words)
