"""Output arrays in pooled pinned memory: results that are kept stay as they
were, views keep their block, released blocks are used again, and past the
bound arrays are ordinary."""
import gc
import os
import threading

import numpy as np
import pytest

from _models import MIX_IDS, hip_cfg, oracle_cfg

pytestmark = pytest.mark.gpu


def test_kept_outputs_stay(hip):
    ocfg = oracle_cfg(n_layers=1, vocab=32000)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS[ocfg.mix], ocfg.seed, ocfg.weight_std)
    dec.observe([1, 2, 3])
    kept, copies = [], []
    for i in range(6):
        rows = dec.batched_logits([i, i + 1])
        dec.rollback_to(3)
        kept.append(rows if i % 2 else rows[1])  # a view alone keeps its block
        copies.append(np.array(kept[-1]))
        rows = None
    for a, b in zip(kept, copies):
        assert np.array_equal(a, b) and a.flags.writeable
    dec.close()


def test_pool_reuse_bound_and_threads(hip):
    pool = hip._PinnedPool()
    a = pool.empty((100, 1000))
    at = a.ctypes.data
    del a
    gc.collect()
    assert pool.empty((100, 1000)).ctypes.data == at
    pool.LIMIT = 1 << 20
    held = [pool.empty(200000) for _ in range(4)]  # 0.8 MB each: one pinned, then ordinary arrays
    assert pool._pinned <= pool.LIMIT
    assert len({h.ctypes.data for h in held}) == 4
    seen = []

    def work(k):
        for i in range(200):
            x = pool.empty(30000)
            x[:] = 1000 * k + i
            seen.append(bool((x == 1000 * k + i).all()))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert len(seen) == 800 and all(seen)


def test_forked_child_reads_results(hip):
    """A kept result in a forked child, handed to write(2): EFAULT where its pages did not come along."""
    ocfg = oracle_cfg(n_layers=1, vocab=32000)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS[ocfg.mix], ocfg.seed, ocfg.weight_std)
    dec.observe([1, 2, 3])
    for _ in range(4):  # results in blocks that were used before, too
        rows = dec.batched_logits([4, 5])
        dec.rollback_to(3)
    r, w = os.pipe()
    pid = os.fork()
    if pid == 0:
        try:
            os.write(w, rows.reshape(-1)[-1000:])
        finally:
            os._exit(0)
    os.close(w)
    with os.fdopen(r, "rb") as f:
        got = np.frombuffer(f.read(), np.float32)
    os.waitpid(pid, 0)
    assert np.array_equal(got, rows.reshape(-1)[-1000:])
    dec.close()
