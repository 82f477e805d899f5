"""hip.Buffer on the CPU, with a runtime that runs out of memory: the memory that the library keeps
from a closed plan is given back before an allocation fails."""
import pytest

import pentago_amd as P
from pentago_amd import hip


class Runtime:
    """hipMalloc fails until `free` is set, as the runtime does, and leaves its error behind."""

    def __init__(self):
        self.free, self.error, self.freed = False, 0, []

    def hipMalloc(self, p, n):
        if not self.free:
            self.error = 2
            return 2
        p._obj.value = 4096
        return 0

    def hipGetLastError(self):
        e, self.error = self.error, 0
        return e

    def hipFree(self, p):
        self.freed.append(p.value)
        return 0

    def hipGetErrorString(self, e):
        return b"out of memory"


@pytest.mark.parametrize("kept", [True, False])
def test_kept_memory_is_given_back_before_an_allocation_fails(monkeypatch, kept):
    runtime = Runtime()
    released = []

    def release():
        released.append(1)
        runtime.free = kept

    monkeypatch.setattr(hip, "_hip", runtime)
    monkeypatch.setattr(P, "release_kept_memory", release, raising=False)
    if kept:
        b = hip.Buffer(100)
        assert b.ptr == 4096 and runtime.error == 0
        del b
        assert runtime.freed == [4096]
    else:
        with pytest.raises(RuntimeError):
            hip.Buffer(100)
    assert released == [1]
