"""The matmul above 16 rows at the edges of its tiles: 32-token tiles and 32-row
groups (128-row workgroups), one superblock of K, odd superblock counts and
inputs one row past a tile, every format, against the kernel's own operands
in f64 (fp16 activations times the emulated fp16 weights)."""
import numpy as np
import pytest

import oracle as O
from _models import MIX_IDS, hip_cfg, oracle_cfg, rel_err
from test_gpu_kernels import operand_weights

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
