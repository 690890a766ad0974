"""Prompts longer than max_batch: chunks of causal rows through the layers (one
forward up to 2048 rows, even shares in whole 128-row blocks beyond, a remainder
of up to 16 rows by itself) against the oracle and against the same tokens observed piece by
piece; the cache rows, the history and what follows the prompt agree too."""
import ctypes

import numpy as np
import pytest

import oracle as O
from _models import MIX_IDS, hip_cfg, oracle_cfg, rel_err

pytestmark = pytest.mark.gpu

LLAMA = dict(n_layers=2, hidden=512, n_heads=8, n_kv_heads=2, head_dim=64, ffn=768, vocab=2048, mix="q4_k_m")
QWEN = dict(arch="qwen2", n_layers=2, hidden=1792, n_heads=14, n_kv_heads=2, head_dim=128, ffn=512, vocab=2048,
            mix="q5k_q80", rope_theta=1e6)


def _dec(hip, ocfg, max_batch):
    d = hip.HipQuantDecoder(hip_cfg(hip, ocfg, max_batch=max_batch))
    d.synthesize(MIX_IDS[ocfg.mix], ocfg.seed, ocfg.weight_std)
    return d


def _kv(d, ocfg, n):
    return np.stack([d.read_kv_rows(li, w, h, 0, n).view(np.float16).astype(np.float64)
                     for li in range(ocfg.n_layers) for w in (0, 1) for h in range(ocfg.n_kv_heads)])


@pytest.mark.parametrize("shape", [LLAMA, QWEN], ids=["llama", "qwen2"])
@pytest.mark.parametrize("before,n,max_batch", [(0, 129, 128), (0, 300, 128), (37, 385, 128), (5, 97, 24), (600, 200, 64)])
def test_prompt_chunks(hip, shape, before, n, max_batch):
    ocfg = oracle_cfg(ctx_len=1024, **shape)
    ids = [int(v) for v in np.random.default_rng(n).integers(0, ocfg.vocab, before + n + 1)]
    a, b = _dec(hip, ocfg, max_batch), _dec(hip, ocfg, 16)
    od = O.OracleDecoder(O.OracleModel(ocfg))
    if before:
        a.observe(ids[:before])
        b.observe(ids[:before])
    a.observe(ids[before:before + n])
    for i in range(before, before + n, 16):  # 16 rows at a time: the kernels of small inputs
        b.observe(ids[i:min(i + 16, before + n)])
    od.observe(ids[:before + n])
    assert a.history() == ids[:before + n] and a.cache_len() == before + n
    ref = od.next_logits()
    assert rel_err(a.next_logits(), ref) < 1e-2
    # two device routes: fp16 activations (and K-quant weights above 16 rows) through 2 layers
    assert rel_err(a.next_logits(), b.next_logits().astype(np.float64)) < 5e-3
    ka, kb = _kv(a, ocfg, before + n), _kv(b, ocfg, before + n)
    assert np.linalg.norm(ka - kb) < 5e-3 * np.linalg.norm(kb)
    assert np.max(np.abs(ka - kb)) < 2e-2 * np.max(np.abs(kb))
    a.observe(ids[-1:])
    od.observe(ids[-1:])
    assert rel_err(a.next_logits(), od.next_logits()) < 1e-2
    a.close()
    b.close()


@pytest.mark.parametrize("before,over", [
    (0, dict(n_heads=4, n_kv_heads=4, mix="q8_0")),
    (45, dict(n_heads=4, n_kv_heads=2, mix="q4_k")),  # grouped KV heads behind a cached prefix
], ids=["mha", "gqa-prefix"])
def test_prompt_beyond_one_chunk(hip, before, over):
    """2113 rows: the even share rounded up to whole 128-row blocks, 1152, then
    961 (and 65 = 2113 % 128 rows stay in them)."""
    ocfg = oracle_cfg(ctx_len=2304, n_layers=1, hidden=256, head_dim=64, ffn=256, vocab=1024, **over)
    ids = [int(v) for v in np.random.default_rng(9).integers(0, ocfg.vocab, before + 2113)]
    a, b = _dec(hip, ocfg, 128), _dec(hip, ocfg, 128)
    if before:
        a.observe(ids[:before])
        b.observe(ids[:before])
    ha = a.observe_returning_last_hidden(ids[before:])
    for i in range(before, len(ids), 100):
        hb = b.observe_returning_last_hidden(ids[i:i + 100])
    assert rel_err(ha, hb.astype(np.float64)) < 5e-3
    ka, kb = _kv(a, ocfg, len(ids)), _kv(b, ocfg, len(ids))
    assert np.linalg.norm(ka - kb) < 5e-3 * np.linalg.norm(kb)
    assert rel_err(a.next_logits(), b.next_logits().astype(np.float64)) < 5e-3
    a.close()
    b.close()


@pytest.mark.parametrize("max_batch,most", [(16, 96 << 20), (128, 512 << 20)])
def test_work_buffers_follow_max_batch(hip, max_batch, most):
    """A handle of up to 16 rows takes prompts in passes of max_batch, and holds
    no buffers for chunks of 2048 rows (at these widths 0.29 GB beside 17 MB of cache)."""
    rt = hip._hip_runtime()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def left():
        assert rt.hipDeviceSynchronize() == 0
        assert rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    ocfg = oracle_cfg(ctx_len=4096, n_layers=1, hidden=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=1024)
    hip.HipQuantDecoder(hip_cfg(hip, ocfg, max_batch=max_batch)).close()  # the library's own allocations
    before = left()
    d = hip.HipQuantDecoder(hip_cfg(hip, ocfg, max_batch=max_batch))
    assert before - left() < most
    d.close()
