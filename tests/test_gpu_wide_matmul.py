"""The matmul above 16 rows at the edges of its tiles: 32-token tiles and 32-row
groups (128-row workgroups), one superblock of K, odd superblock counts and
inputs one row past a tile, every format, against the kernel's own operands
in f64 (fp16 activations times the emulated fp16 weights)."""
import types

import numpy as np
import pytest

import oracle as O
from _models import MIX_IDS, hip_cfg, oracle_cfg, rel_err
from test_gpu_kernels import operand_weights
from test_zz_no_alloc import DevBuf, _hip_runtime, _noalloc

pytestmark = pytest.mark.gpu

# 64, 256, 768 and 288 rows of K 256 and 256 rows of K 768: less than a
# workgroup's rows, whole ones, a last one with a single 32-row group
SHAPE = dict(n_layers=1, hidden=256, n_heads=4, n_kv_heads=1, head_dim=64, ffn=768, vocab=288, ctx_len=64)
KINDS = (O.K_ATTN_K, O.K_ATTN_Q, O.K_FFN_UP, O.K_FFN_DOWN, O.K_OUTPUT)


@pytest.mark.parametrize("mix", ["q4_k", "q5_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("M", [17, 31, 32, 33, 63, 65, 95, 96, 97, 127])
def test_tile_edges(hip, mix, M):
    ocfg = oracle_cfg(mix=mix, **SHAPE)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS[mix], ocfg.seed, ocfg.weight_std)
    for kind in KINDS:
        layer = -1 if kind == O.K_OUTPUT else 0
        fmt, raw = O.synth_tensor(ocfg, layer, kind)
        rows, K = ocfg.shape(kind)
        x = np.random.default_rng(M * 31 + kind).standard_normal((M, K)).astype(np.float32)
        y = dec.qmatmul(layer, kind, x)
        ref = O.round_f16(x).astype(np.float64) @ operand_weights(fmt, raw, rows, K, M).astype(np.float64).T
        # f32 sums of K exact products: at most K ulps of the sum of magnitudes, far below in practice
        assert rel_err(y, ref) < K * 2.0 ** -24 * 8, (kind, rel_err(y, ref))
    dec.close()


def test_noalloc_split_unaligned_rows(hip):
    """The allocation-free product with K slices (256 output rows, K = 7168: seven
    or eight slices) on inputs and outputs that start one float into an allocation."""
    ocfg = oracle_cfg(mix="q4_k", n_layers=1, hidden=256, n_heads=4, n_kv_heads=1, head_dim=64, ffn=7168, vocab=256,
                      ctx_len=64)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS["q4_k"], ocfg.seed, ocfg.weight_std)
    rows, K = ocfg.shape(O.K_FFN_DOWN)
    rt = _hip_runtime()
    for M in (17, 40, 128):
        x = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
        exp = dec.qmatmul(0, O.K_FFN_DOWN, x)
        for at in (0, 1):
            xb, yb = DevBuf(rt, 4 * (M * K + 4)), DevBuf(rt, 4 * (M * rows + 4))
            xb.put(np.concatenate([np.zeros(at, np.float32), x.reshape(-1)]))
            yb.put(np.zeros(M * rows + 4, np.float32))
            xo, yo = types.SimpleNamespace(p=xb.p.value + 4 * at), types.SimpleNamespace(p=yb.p.value + 4 * at)
            assert _noalloc(hip, dec, 0, O.K_FFN_DOWN, xo, M, yo) == 0
            dec.synchronize()
            got = yb.get(M * rows + 4)
            assert np.array_equal(got[at:at + M * rows].view(np.uint32), exp.reshape(-1).view(np.uint32)), (M, at)
            assert not got[at + M * rows:].any()
            xb.free()
            yb.free()
    dec.close()


@pytest.mark.parametrize("M", [5, 17, 40, 128])
def test_noalloc_unsplit_unaligned_rows(hip, M):
    """One superblock of K: the product's own stores write the caller's rows,
    which start 0 to 3 floats into an allocation."""
    ocfg = oracle_cfg(mix="q4_k", **SHAPE)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS["q4_k"], ocfg.seed, ocfg.weight_std)
    rt = _hip_runtime()
    for kind in (O.K_ATTN_Q, O.K_FFN_UP):
        rows, K = ocfg.shape(kind)
        x = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
        exp = dec.qmatmul(0, kind, x)
        xb, yb = DevBuf(rt, 4 * M * K), DevBuf(rt, 4 * (M * rows + 8))
        xb.put(x)
        for at in range(4):
            yb.put(np.zeros(M * rows + 8, np.float32))
            yo = types.SimpleNamespace(p=yb.p.value + 4 * at)
            assert _noalloc(hip, dec, 0, kind, xb, M, yo) == 0
            dec.synchronize()
            got = yb.get(M * rows + 8)
            assert np.array_equal(got[at:at + M * rows].view(np.uint32), exp.reshape(-1).view(np.uint32)), (kind, at)
            assert not got[:at].any() and not got[at + M * rows:].any()
        xb.free()
        yb.free()
    dec.close()


@pytest.mark.parametrize("mix", ["q4_k", "q5_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("M", [33, 47, 64])
def test_more_workgroups_than_cus(hip, mix, M):
    """33 to 64 rows of more than 256 128-row blocks (257 here, the last one a
    single 32-row group) take four-wave workgroups: the plain product, and in a
    tree pass the lm_head with its argmax and gate/up (260 blocks)."""
    ocfg = oracle_cfg(mix=mix, **dict(SHAPE, ffn=16640, vocab=32800, ctx_len=128))
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS[mix], ocfg.seed, ocfg.weight_std)
    fmt, raw = O.synth_tensor(ocfg, -1, O.K_OUTPUT)
    rows, K = ocfg.shape(O.K_OUTPUT)
    x = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    ref = O.round_f16(x).astype(np.float64) @ operand_weights(fmt, raw, rows, K, M).astype(np.float64).T
    assert rel_err(dec.qmatmul(-1, O.K_OUTPUT, x), ref) < K * 2.0 ** -24 * 8
    prefix = [5, 6, 7]
    toks = [7] + [int(v) for v in np.random.default_rng(M).integers(0, ocfg.vocab, M - 1)]
    tree = (toks, [0] + [max(0, (i - 1) // 3) for i in range(1, M)])
    dec.observe(prefix)
    logits, hidden = dec.tree_logits_keep_kv(tree)
    best = dec.last_argmax(M)
    assert np.array_equal(best, logits.argmax(1))
    # the same nodes one root path at a time, on the kernels of up to 16 rows
    path = []
    i = M - 1
    while i:
        path.append(i)
        i = tree[1][i]
    dec.rollback_to(len(prefix))
    step = dec.batched_logits([toks[j] for j in path[::-1]])
    # fp16 activations and K-quant weights against exact-integer weights, through one layer
    assert rel_err(logits[[0] + path[::-1]], step.astype(np.float64)) < 5e-3
    dec.close()


def test_small_launches_above_64_rows(hip):
    """65 to 128 rows of launches that leave most CUs idle take two token tiles
    a workgroup, with and without K slices."""
    ocfg = oracle_cfg(mix="q4_k", n_layers=1, hidden=512, n_heads=8, n_kv_heads=8, head_dim=64, ffn=1536, vocab=288,
                      ctx_len=64)
    dec = hip.HipQuantDecoder(hip_cfg(hip, ocfg))
    dec.synthesize(MIX_IDS["q4_k"], ocfg.seed, ocfg.weight_std)
    for kind in (O.K_ATTN_Q, O.K_FFN_UP, O.K_FFN_DOWN):
        fmt, raw = O.synth_tensor(ocfg, 0, kind)
        rows, K = ocfg.shape(kind)
        for M in (65, 97, 128):
            x = np.random.default_rng(M + kind).standard_normal((M, K)).astype(np.float32)
            ref = O.round_f16(x).astype(np.float64) @ operand_weights(fmt, raw, rows, K, M).astype(np.float64).T
            assert rel_err(dec.qmatmul(0, kind, x), ref) < K * 2.0 ** -24 * 8, (kind, M)
    dec.close()
