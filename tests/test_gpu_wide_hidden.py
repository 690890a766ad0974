"""Hidden sizes above 4096: the RMSNorm kernels of two and four vectors a thread
and the strided one, with and without K slices to add, and the passes of up to
16 rows whose norms are launches of their own at these widths."""
import numpy as np
import pytest

import oracle as O
from _models import MIX_IDS, hip_cfg, oracle_cfg, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-2  # logits and hidden states against the oracle, as for the other decoders


# 4608 and 5120: two vectors a thread, 9216: four, 8448 (a multiple of 256 alone): strided
@pytest.mark.parametrize("hidden,kv_heads", [(4608, 4), (5120, 8), (9216, 8), (8448, 2)])
def test_hidden_widths(hip, hidden, kv_heads):
    ocfg = oracle_cfg(n_layers=1, hidden=hidden, n_heads=hidden // 128, n_kv_heads=kv_heads, head_dim=128, ffn=2048,
                      vocab=512, ctx_len=512)
    od = O.OracleDecoder(O.OracleModel(ocfg))
    hd = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    hd.synthesize(MIX_IDS[ocfg.mix], ocfg.seed, ocfg.weight_std)
    ids = [int(v) for v in np.random.default_rng(hidden).integers(0, ocfg.vocab, 200)]
    at = 0
    for n in (20, 1, 90):  # 17 to 64 rows, one row, more than 64
        od.observe(ids[at:at + n])
        hd.observe(ids[at:at + n])
        at += n
        assert rel_err(hd.next_logits(), od.next_logits()) < TOL, n
    a, b = hd.batched_logits(ids[at:at + 4]), od.batched_logits(ids[at:at + 4])
    for i in range(5):
        assert rel_err(a[i], b[i]) < TOL, i
    od.rollback_to(at)
    hd.rollback_to(at)
    for n in (9, 24, 70):
        tree = O.DraftTree([ids[at - 1]] + ids[at:at + n - 1], [0] + [(i - 1) // 2 for i in range(1, n)])
        la, ha = hd.tree_logits_keep_kv((tree.tokens(), tree.parents()))
        lb, hb = od.tree_logits_keep_kv(tree)
        assert rel_err(la, lb) < TOL and rel_err(ha, hb) < TOL, n
        od.rollback_to(at)
        hd.rollback_to(at)
    # the last row's norm alone, after up to 16, up to 64 and more rows
    for n in (7, 33, 80):
        h = hd.observe_returning_last_hidden(ids[at:at + n])
        at_one = hd.last_hidden_state()  # the same row as a pass of its own
        assert rel_err(h, at_one.astype(np.float64)) < TOL, n
        hd.rollback_to(at)
    hd.close()
