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
        self.refuse, self.last, self.allocs, self.blocks, self.pool = refuse, 0, 0, {}, None

    def hipHostMalloc(self, out, size, flags):
        self.allocs += 1
        assert not (self.pool and self.pool._lock.locked()), "an allocation with the lock held"
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
        assert not (self.pool and self.pool._lock.locked()), "a free with the lock held"
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
    for _ in range(2):
        a, b = pool.empty((64, 1000)), pool.empty(70000)
        pool.grow()
    assert runtime.allocs == 2 and not a.flags.owndata
    a[:], b[:] = 3.5, -1.0
    view, gone = a[5], pool.empty((300, 1000))
    del a, gone
    pool.RETAIN = 0

    def probe():
        nonlocal b
        ok = (view == 3.5).all() and (b == -1.0).all() and pool.empty((64, 1000)).flags.owndata
        view[:] = 9.0
        b = None  # a carried-over block that comes back is not the child's to free
        pool.acquire()
        pool.release()
        ok = ok and len(runtime.blocks) == 2
        return b"same" if ok else b"other"

    try:
        assert _forked(probe) == b"same"
        assert (view == 3.5).all() and pool.LIMIT > 0
        del b
        assert not pool.empty(70000).flags.owndata  # the parent's pool goes on
    finally:
        del pool.RETAIN
        for d in (pool._free, pool._used, pool._count, pool._want):
            d.clear()
        pool._pinned = 0


def test_results_never_wait_for_an_allocation(runtime):
    pool = runtime.pool = S._PinnedPool(deferred=True)
    first = pool.empty((5, 32000))
    assert runtime.allocs == 0 and first.flags.owndata
    pool.grow()
    assert runtime.allocs == 1
    a = pool.empty((5, 32000))
    assert not a.flags.owndata and runtime.allocs == 1
    at = a.ctypes.data
    del a
    assert pool.empty((4, 32000)).ctypes.data == at  # a block serves smaller results too
    pool.grow()
    assert runtime.allocs == 1  # and nothing is wanted


def test_a_caller_that_keeps_results(runtime):
    """At most two blocks of a size per open decoder, then ordinary arrays."""
    pool = runtime.pool = S._PinnedPool(deferred=True)
    for users in (1, 2):
        pool.acquire()
        kept = []
        for _ in range(8):
            kept.append(pool.empty(100000))
            pool.grow()
        assert sum(not k.flags.owndata for k in kept) == 2 * users == runtime.allocs
        assert len({k.ctypes.data for k in kept}) == 8
        del kept


def test_free_blocks_are_given_back_with_the_last_decoder(runtime):
    pool = runtime.pool = S._PinnedPool(deferred=True)
    pool.RETAIN = 1 << 20
    pool.acquire()
    pool.acquire()
    for n in (50000, 150000, 300000):
        pool.empty(n)
        pool.grow()
    kept = pool.empty(50000)
    kept[:] = 2.0
    pool.release()
    assert len(runtime.blocks) == 3
    pool.release()
    assert len(runtime.blocks) == 2 and (kept == 2.0).all()  # one kept by the caller, one within RETAIN
    assert pool._pinned == pool._size(kept.nbytes) + pool._size(4 * 150000) == sum(map(len, runtime.blocks.values()))
    del kept
    pool.acquire()
    assert not pool.empty(150000).flags.owndata
    pool.RETAIN = 0
    pool.release()
    assert not runtime.blocks and pool._pinned == 0


@pytest.mark.parametrize("deferred", [False, True])
def test_bound(runtime, deferred):
    pool = runtime.pool = S._PinnedPool(deferred=deferred)
    pool.LIMIT = 1 << 20
    kept = []
    for n in (30000, 60000, 90000, 120000, 150000, 180000):
        for _ in range(3):
            kept.append(pool.empty(n))
            pool.grow()
            assert pool._pinned <= pool.LIMIT and pool._pinned == sum(map(len, runtime.blocks.values()))
    assert len({k.ctypes.data for k in kept}) == len(kept)


def test_size_classes():
    pool = S._PinnedPool()
    for n in list(range(1, 3 << 20, 4099)) + [128 * 152064 * 4]:
        s = pool._size(n)
        assert n <= s <= max(n * 1.25 + pool.GRAIN, pool.GRAIN) and s % pool.GRAIN == 0
