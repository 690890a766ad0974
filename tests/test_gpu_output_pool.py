"""Output arrays in pooled pinned memory: results that are kept stay as they
were, views keep their block, released blocks are used again, and past the
bound arrays are ordinary."""
import gc
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
