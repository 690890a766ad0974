"""The pool of pinned output arrays on the CPU: a stand-in for the HIP runtime
hands out anonymous pages that, like the driver's, a forked child does not get."""
import ctypes
import mmap

import numpy as np
import pytest

import speculate_hip as S


class Runtime:
    """hipHostMalloc and its neighbours over anonymous memory; `refuse` makes
    allocations fail, `last` is the thread's sticky error."""

    def __init__(self, refuse=False):
        self.refuse, self.last, self.allocs, self.blocks = refuse, 0, 0, {}

    def hipHostMalloc(self, out, size, flags):
        self.allocs += 1
        if self.refuse:
            self.last = 2
            return 2
        m = mmap.mmap(-1, size)
        m.madvise(mmap.MADV_DONTFORK)
        at = ctypes.addressof(ctypes.c_char.from_buffer(m))
        self.blocks[at] = m
        out._obj.value = at
        return 0

    def hipHostFree(self, p):
        assert self.blocks.pop(p.value, None) is not None, "freed twice, or never allocated"
        return 0

    def hipGetLastError(self):
        e, self.last = self.last, 0
        return e


@pytest.fixture
def runtime(monkeypatch):
    rt = Runtime()
    monkeypatch.setattr(S, "_hip_runtime", lambda: rt)
    return rt


def test_refused_allocation_leaves_no_error(runtime):
    runtime.refuse = True
    pool = S._PinnedPool()
    a = pool.empty((100, 1000))
    assert runtime.allocs == 1 and a.flags.owndata and a.shape == (100, 1000)
    assert pool._pinned == 0 and runtime.last == 0
