"""The pool of pinned output arrays on the CPU: a stand-in for the HIP runtime
hands out anonymous pages that, like the driver's, a forked child does not get."""
import ctypes
import mmap
import os

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


def _forked(probe) -> bytes:
    """What probe() returns in a forked child (b"" if the child died)."""
    r, w = os.pipe()
    pid = os.fork()
    if pid == 0:
        try:
            os.write(w, probe())
        finally:
            os._exit(0)
    os.close(w)
    got = os.read(r, 4096)
    os.close(r)
    os.waitpid(pid, 0)
    return got


def test_results_are_readable_in_a_forked_child(runtime):
    """Kept results and views read the same in a child, whose own results are
    ordinary; the parent's stay shared with nobody."""
    pool = S._pinned  # the one whose fork hooks are registered
    a, b = pool.empty((64, 1000)), pool.empty(70000)
    assert runtime.allocs == 2 and not a.flags.owndata
    a[:], b[:] = 3.5, -1.0
    view, gone = a[5], pool.empty((300, 1000))
    del a, gone

    def probe():
        ok = (view == 3.5).all() and (b == -1.0).all() and pool.empty((64, 1000)).flags.owndata
        view[:] = 9.0
        return b"same" if ok else b"other"

    try:
        assert _forked(probe) == b"same"
        assert (view == 3.5).all() and pool.LIMIT > 0
        c = pool.empty((64, 1000))  # the parent's pool goes on
        assert not c.flags.owndata
    finally:
        pool._free.clear()
        pool._used.clear()
        pool._pinned = 0
