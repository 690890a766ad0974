// K1 above 16 rows (tree verification, prompts): y[m][n] = sum_k x[m][k] * W[n][k]
// on v_mfma_f32_32x32x16_f16, weights dequantised to fp16 in registers.
//
// A workgroup owns 128 rows (4 row groups of 32) and TT token tiles of 32, for
// one K slice.  KH = 2: two waves share a row group, wave half kh multiplies
// K-chunks 4 kh .. 4 kh + 3 of every superblock, so a SIMD holds two waves
// (one's dequantisation runs behind the other's MFMAs) and no weight is
// fetched or dequantised twice; the halves' sums meet in LDS at the end.
// KH = 1: a wave of its own per row group, and a SIMD's two waves come from two
// workgroups, for launches of more workgroups than CUs (wide_kh).
// Activations arrive in operand order (xt_index, sd_common.hpp): a superblock
// of a token tile is 16 KiB of MFMA operands, 1 KiB each in lane order, so the
// copy to LDS and every LDS read are contiguous and free of bank conflicts.
//
// What bounds it: per 32-row tile, token tile and superblock 16 MFMAs (17 ns
// each with the whole chip busy, when it clocks at 1.9 GHz) against about 17
// other vector instructions per MFMA step (2 ns each), which issue beside
// another wave's MFMAs but not beside their own wave's: instruction issue up to
// 64 rows (a superblock of 128 rows and 64 tokens takes 0.9 us with 64
// workgroups running, 1.0 with 256, its MFMAs 0.55), the MFMAs most of it above
// (128 tokens: 1.3 us with 128 workgroups, 1.5 with 256 and 1.65 for Q6_K and
// Q8_0, against 1.09).  A launch adds 4 to 9 us, the more the more it stores (9
// with 17 MB of outputs).  Gate/up of 2 x 14336 x 4096
// Q4_K (weights in the caches) at 27 / 60 / 128 rows: 18.7 / 21.5 / 32.2 us,
// where one 16-row tile per wave with the activations in row order took
// 23.8 / 33.1 / 55.7 us; at 512 rows 148 us (812 TFLOP/s).
//
// Dequantisation to fp16: a code is OR'ed into the mantissa of 1024.0h
// (0x6400 | q == 1024 + q) or, for a code already at bits 4-7, of 64.0h
// (0x5400 | q << 4 == 64 + q); the offset is subtracted exactly and one packed
// fp16 operation applies the scale (Q6_K: fp16(d * sc); Q8_0: d) or the scale
// and min (Q4_K / Q5_K: round_f16(q * s16 - m16), s16 = fp16(d * sc), m16 =
// fp16(dmin * m)).  The sub-block scales are formed in packed fp16 (d * sc of
// an exact integer sc rounds once) and broadcast by operand selects.
#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>

#include "sd_buffer.hpp"
#include "sd_common.hpp"
#include "sd_kernels.hpp"
#include "sd_qcodes.hpp"

namespace sd {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ half2v h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t u2(half2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2v lo2(half2v v) { return half2v{v.x, v.x}; }
__device__ __forceinline__ half2v hi2(half2v v) { return half2v{v.y, v.y}; }
__device__ __forceinline__ half8 cat8(half2v a, half2v b, half2v c, half2v d) {
    const uintx4 u = {u2(a), u2(b), u2(c), u2(d)};
    return __builtin_bit_cast(half8, u);
}
constexpr uint32_t kM1024 = 0xE400E400u, kM64 = 0xD400D400u;      // (-1024, -1024), (-64, -64) in fp16
constexpr uint32_t kM1056 = 0xE420E420u, kM96 = 0xD600D600u;      // (-1056, ..), (-96, ..)
constexpr uint32_t kM1152 = 0xE480E480u;                          // (-1152, ..)

// N dwords (1, 2 or 4) at lane offset vo, uniform offset so
template <int N> struct Dw {
    uint32_t w[N];
};
template <int N> __device__ __forceinline__ Dw<N> bldn(rsrc_t rs, uint32_t vo, uint32_t so) {
    if constexpr (N == 4) return __builtin_bit_cast(Dw<4>, bld16(rs, vo, so));
    else if constexpr (N == 2) return __builtin_bit_cast(Dw<2>, bld8(rs, vo, so));
    else return Dw<1>{{bld4(rs, vo, so)}};
}

// --------------------------------------------------------------------------
// One lane's share of a 32-row tile and superblock.  Lane (r = lane & 31, j = lane >> 5) holds row r; MFMA
// step 2 c + p of chunk c takes the 8 codes of (row, lane group g = j + 2 p)
// that the 16-row layout gives lane (row & 15) + 16 g of the row's tile block.
// vo: the row's tile block (a lane offset); so: the superblock (uniform); kh:
// the wave's half of the superblock's chunks.
// --------------------------------------------------------------------------
template <int FMT> struct WFmt;

// scale pair {s, -m} of the two sub-blocks of a lane group
struct KScale {
    half2v a, b;
};
__device__ __forceinline__ KScale kq_scale(const Dw<4> &hdr, int g) {
    // w = sc_2g | sc_2g+1 << 6 | m_2g << 12 | m_2g+1 << 18 (kq_hdr_pack)
    const uint32_t lo = __builtin_amdgcn_perm(hdr.w[2], hdr.w[1], 0x0c0c0000u | (uint32_t)(4 + g) << 8 | (uint32_t)g);
    const uint32_t w = __builtin_amdgcn_perm(hdr.w[3], lo, 0x0c000100u | (uint32_t)(4 + g) << 16);
    const uint32_t a = 0x64006400u | (w & 0x3fu) | ((w & 0x3f000u) << 4);
    const uint32_t b = 0x64006400u | ((w >> 6) & 0x3fu) | (((w >> 6) & 0x3f000u) << 4);
    const half2v d = h2(hdr.w[0] ^ 0x80000000u);  // {d, -dmin}
    KScale k;
    k.a = (h2(a) + h2(kM1024)) * d;
    k.b = (h2(b) + h2(kM1024)) * d;
    return k;
}
// codes -> round_f16(q * s - m)
__device__ __forceinline__ half2v kq(uint32_t p, uint32_t off, half2v sm) {
    return __builtin_elementwise_fma(h2(p) + h2(off), lo2(sm), hi2(sm));
}

template <> struct WFmt<Q4_K> {
    static constexpr int TBB = LaneQ4K::TBB;
    struct D {
        Dw<4> hdr;
        Dw<4> q[2];
    };
    typedef KScale S[2];
    static __device__ __forceinline__ void load(D &d, rsrc_t rs, uint32_t vo, uint32_t so, int r, int j, int kh) {
        d.hdr = bldn<4>(rs, vo + (r & 15) * 16, so);
#pragma unroll
        for (int p = 0; p < 2; p++)
            d.q[p] = bldn<4>(rs, vo + 256 + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 1024);
    }
    static __device__ __forceinline__ void scales(const D &d, S &s, int j, int kh) {
        s[0] = kq_scale(d.hdr, j);
        s[1] = kq_scale(d.hdr, j + 2);
    }
    static __device__ __forceinline__ half8 frag(const D &d, const S &s, int c, int p) {
        const uint32_t w = d.q[p].w[c], w8 = w >> 8, e64 = 0x64006400u, e54 = 0x54005400u;
        return cat8(kq(and_or(w, 0x000F000Fu, e64), kM1024, s[p].a), kq(and_or(w8, 0x000F000Fu, e64), kM1024, s[p].a),
                    kq(and_or(w, 0x00F000F0u, e54), kM64, s[p].b), kq(and_or(w8, 0x00F000F0u, e54), kM64, s[p].b));
    }
};

template <> struct WFmt<Q5_K> {
    static constexpr int TBB = LaneQ5K::TBB;
    struct D {
        Dw<4> hdr;
        Dw<4> q[2];
        uint32_t qh[2];
    };
    typedef KScale S[2];
    static __device__ __forceinline__ void load(D &d, rsrc_t rs, uint32_t vo, uint32_t so, int r, int j, int kh) {
        d.hdr = bldn<4>(rs, vo + (r & 15) * 16, so);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            d.qh[p] = bld4(rs, vo + 256 + ((r & 15) + 16 * j) * 8 + p * 256, so + kh * 4);
            d.q[p] = bldn<4>(rs, vo + 768 + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 1024);
        }
    }
    static __device__ __forceinline__ void scales(const D &d, S &s, int j, int kh) {
        s[0] = kq_scale(d.hdr, j);
        s[1] = kq_scale(d.hdr, j + 2);
    }
    static __device__ __forceinline__ half8 frag(const D &d, const S &s, int c, int p) {
        const uint32_t w = d.q[p].w[c], w8 = w >> 8;
        const uint32_t R = rotr(d.qh[p], LaneQ5K::rot(c)), R1 = R >> 1;
        const uint32_t x02 = and_or(R, 0x00100010u, 0x64006400u), x13 = and_or(R1, 0x00100010u, 0x64006400u);
        const uint32_t y02 = and_or(R, 0x01000100u, 0x54005400u), y13 = and_or(R1, 0x01000100u, 0x54005400u);
        return cat8(kq(and_or(w, 0x000F000Fu, x02), kM1024, s[p].a), kq(and_or(w8, 0x000F000Fu, x13), kM1024, s[p].a),
                    kq(and_or(w, 0x00F000F0u, y02), kM64, s[p].b), kq(and_or(w8, 0x00F000F0u, y13), kM64, s[p].b));
    }
};

template <> struct WFmt<Q6_K> {
    static constexpr int TBB = LaneQ6K::TBB;
    struct D {
        Dw<4> n[2];
        Dw<2> hb[2];
        uint32_t sc[2], d;
    };
    typedef half2v S[2];  // {d * sc(s' = 0), d * sc(s' = 1)} of the chunk half
    static __device__ __forceinline__ void load(D &d, rsrc_t rs, uint32_t vo, uint32_t so, int r, int j, int kh) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            d.n[p] = bldn<4>(rs, vo + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 1024);
            d.hb[p] = bldn<2>(rs, vo + 2048 + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 8);
            d.sc[p] = bld4(rs, vo + 3072 + (r & 15) * 16 + 4 * j + 8 * p, so);
        }
        d.d = bld2(rs, vo + 3328 + (r & 15) * 2, so);
    }
    static __device__ __forceinline__ void scales(const D &d, S &s, int j, int kh) {
        const half2v dd = h2(d.d * 0x10001u);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            // bytes kh and 2 + kh of the lane group's scales, + 128, in the 1024 binade
            const uint32_t v = ((d.sc[p] >> (8 * kh)) & 0x00ff00ffu) ^ 0x64806480u;
            s[p] = (h2(v) + h2(kM1152)) * dd;
        }
    }
    static __device__ __forceinline__ half8 frag(const D &d, const S &s, int c, int p) {
        const uint32_t w = d.n[p].w[c], w8 = w >> 8;
        const uint32_t R = rotr(d.hb[p].w[c >> 1], 8 * (c & 1)), R2 = R >> 2;
        const uint32_t x02 = and_or(R, 0x00300030u, 0x64006400u), x13 = and_or(R2, 0x00300030u, 0x64006400u);
        const uint32_t y02 = and_or(R, 0x03000300u, 0x54005400u), y13 = and_or(R2, 0x03000300u, 0x54005400u);
        return cat8((h2(and_or(w, 0x000F000Fu, x02)) + h2(kM1056)) * lo2(s[p]),
                    (h2(and_or(w8, 0x000F000Fu, x13)) + h2(kM1056)) * lo2(s[p]),
                    (h2(and_or(w, 0x00F000F0u, y02)) + h2(kM96)) * hi2(s[p]),
                    (h2(and_or(w8, 0x00F000F0u, y13)) + h2(kM96)) * hi2(s[p]));
    }
};

template <> struct WFmt<Q8_0> {
    static constexpr int TBB = LaneQ80::TBB;
    struct D {
        Dw<4> a[2], b[2];
        uint32_t d[2];
    };
    typedef half2v S[2];  // {d of block 2g, d of block 2g + 1}
    static __device__ __forceinline__ void load(D &d, rsrc_t rs, uint32_t vo, uint32_t so, int r, int j, int kh) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            d.a[p] = bldn<4>(rs, vo + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 1024);
            d.b[p] = bldn<4>(rs, vo + 2048 + ((r & 15) + 16 * j) * 16 + p * 512, so + kh * 1024);
            d.d[p] = bld4(rs, vo + 4096 + (r & 15) * 16 + 4 * j + 8 * p, so);
        }
    }
    static __device__ __forceinline__ void scales(const D &d, S &s, int j, int kh) {
        s[0] = h2(d.d[0]);
        s[1] = h2(d.d[1]);
    }
    static __device__ __forceinline__ half8 frag(const D &d, const S &s, int c, int p) {
        const uint32_t qa = d.a[p].w[c], qb = d.b[p].w[c], M = 0x64646464u;
        return cat8((h2(perm(qa, M, 0x00060004u)) + h2(kM1152)) * lo2(s[p]),
                    (h2(perm(qa, M, 0x00070005u)) + h2(kM1152)) * lo2(s[p]),
                    (h2(perm(qb, M, 0x00060004u)) + h2(kM1152)) * hi2(s[p]),
                    (h2(perm(qb, M, 0x00070005u)) + h2(kM1152)) * hi2(s[p]));
    }
};

// --------------------------------------------------------------------------
// The main loop
// --------------------------------------------------------------------------
constexpr int kRG = 4;                       // row groups (32 rows each) of a workgroup
constexpr int wide_threads(int KH) { return KH * kRG * 64; }  // KH waves share a row group
constexpr int kXTile = 16384;                // bytes of one token tile's superblock (16 operands of 1 KiB)

struct WideWave {
    rsrc_t w;           // the row tile's matrix
    uint32_t wvo;       // the row's tile block at superblock 0 (lane offset)
    rsrc_t x;
    uint32_t xtile[4];  // the token tiles' offsets
    int sb0, n;         // the slice's superblocks
    int r, j, kh;
};

template <int FMT, int TT, int KH>
__device__ __forceinline__ void wide_body(const WideWave &W, floatx16 (&acc)[TT], uint8_t *lds) {
    typedef WFmt<FMT> F;
    constexpr int STAGE = TT * kXTile;
    constexpr int PIECE = wide_threads(KH) * 16, PT = kXTile / PIECE;  // bytes of a piece, pieces of a token tile
    constexpr int HW = 2 / KH, NS = 8 * HW;                            // chunk halves and MFMA steps of a wave
    const int tid = threadIdx.x, lane = tid & 63;
    const int n = W.n;
    uintx4 xs[PT * TT];
    typename F::D w[2][HW];
    // superblocks past the last are read as the last and not multiplied
    auto ldx = [&](int i, int k) {  // piece k of superblock i's activations
        const uint32_t so = (uint32_t)(min(i, n - 1) + W.sb0) * kXTile;
        xs[k] = bld16(W.x, (uint32_t)tid * 16u, uni(W.xtile[k / PT] + so + (uint32_t)(k % PT) * PIECE));
    };
    auto ldw = [&](typename F::D (&d)[HW], int i) {
#pragma unroll
        for (int h = 0; h < HW; h++)
            F::load(d[h], W.w, W.wvo, uni((uint32_t)(min(i, n - 1) + W.sb0) * F::TBB), W.r, W.j, KH == 2 ? W.kh : h);
    };
    auto put = [&](int i, int k) { *(uintx4 *)(lds + (i & 1) * STAGE + tid * 16 + k * PIECE) = xs[k]; };
    // Superblock i is multiplied; between its MFMA steps, a piece at a time, the
    // activations of i + 1 go to the other LDS stage (every wave is past its
    // reads of i - 1 there) and those of i + 2 are requested.  All at the
    // step's start, the copies held the MFMAs up: ffn_down at 128 rows 95 us,
    // 78 so.
    auto step = [&](const typename F::D (&d)[HW], int i) {
        const uint8_t *xb = lds + (i & 1) * STAGE + (KH == 2 ? W.kh * 8192 : 0) + lane * 16;
        typename F::S sc;
        F::scales(d[0], sc, W.j, KH == 2 ? W.kh : 0);
        half8 b[2][TT], a[2];
#pragma unroll
        for (int tt = 0; tt < TT; tt++) b[0][tt] = *(const half8 *)(xb + tt * kXTile);
        a[0] = F::frag(d[0], sc, 0, 0);
#pragma unroll
        for (int ks = 0; ks < NS; ks++) {
            if (ks < NS - 1) {
                const int kn = ks + 1, h = kn >> 3;
#pragma unroll
                for (int tt = 0; tt < TT; tt++) b[kn & 1][tt] = *(const half8 *)(xb + tt * kXTile + kn * 1024);
                if (kn == 8) F::scales(d[h], sc, W.j, 1);
                a[kn & 1] = F::frag(d[h], sc, (kn & 7) >> 1, kn & 1);
            }
            if (ks % (4 / TT) == 0) {
                put(i + 1, ks / (4 / TT));
                ldx(i + 2, ks / (4 / TT));
            }
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
                acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks & 1], b[ks & 1][tt], acc[tt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The loads' order is pinned: a wait on one load waits for every older one,
    // and the compiler's wait counts are exact only if the order before the
    // loop is the order inside it.
#define PIN __builtin_amdgcn_sched_barrier(0)
#pragma unroll
    for (int k = 0; k < PT * TT; k++) ldx(0, k);
    PIN;
    ldw(w[0], 0);
    PIN;
#pragma unroll
    for (int k = 0; k < PT * TT; k++) put(0, k);
    PIN;
#pragma unroll
    for (int k = 0; k < PT * TT; k++) ldx(1, k);
    PIN;
    ldw(w[1], 1);
    PIN;
    __syncthreads();
    for (int i = 0;; i += 2) {
        step(w[0], i);
        PIN;
        if (i + 1 >= n) return;
        ldw(w[0], i + 2);
        PIN;
        __syncthreads();
        step(w[1], i + 1);
        PIN;
        if (i + 2 >= n) return;
        ldw(w[1], i + 3);
        PIN;
        __syncthreads();
    }
#undef PIN
}

__device__ __forceinline__ float silu_w(float g) { return g / (1.0f + __expf(-g)); }

// The launch's row groups: 32 rows of a segment, or (gate/up) alternating 32
// gate rows and the 32 up rows of the same features.
__host__ __device__ inline int wide_groups(const GemmParams &p) {
    return p.mode == GM_SWIGLU ? p.seg[0].rows / 16 : p.ntiles / 2;
}
// bytes of LDS: two stages of activations, or the sums of two token tiles
constexpr int kYPitch = 36;                         // floats per token of a 32-row tile (conflict free)
constexpr int kYTile = 32 * kYPitch;
template <int TT, int KH> constexpr int wide_lds() {
    const int x = 2 * TT * kXTile, y = KH * kRG * (TT < 2 ? TT : 2) * kYTile * 4;
    return x > y ? x : y;
}

__device__ __forceinline__ void amax_merge(float &bv, int &bi, float ov, int oi) {
    if (oi != 0x7fffffff && (ov > bv || (ov == bv && oi < bi) || bi == 0x7fffffff)) {
        bv = ov;
        bi = oi;
    }
}

struct WideArgs {
    GemmParams g;
    int nrb, nks, ntb;
};

// nrb row blocks x nks K slices x ntb token blocks; workgroups of one (row
// block, slice) sit on one XCD one after the other, so the weights leave HBM
// once and the other token blocks find them in that XCD's L2
template <int TT, int KH, int WPE>
__global__ __launch_bounds__(wide_threads(KH)) __attribute__((amdgpu_waves_per_eu(WPE))) void k_qwide(WideArgs) {
    constexpr int NT = wide_threads(KH);
    warm_kernargs<sizeof(WideArgs)>();
    const GemmParams &p = kernarg<GemmParams, offsetof(WideArgs, g)>();
    const int nrb = kernarg<int, offsetof(WideArgs, nrb)>(), nks = kernarg<int, offsetof(WideArgs, nks)>(),
              ntb = kernarg<int, offsetof(WideArgs, ntb)>();
    extern __shared__ __attribute__((aligned(16))) uint8_t wlds[];
    const int unit = ((int)blockIdx.x >> 3) / ntb * 8 + ((int)blockIdx.x & 7), tblk = ((int)blockIdx.x >> 3) % ntb;
    if (unit >= nrb * nks) return;
    const int rb = unit / nks, ks = unit % nks;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool swi = p.mode == GM_SWIGLU;
    const int nsb = p.K >> 8, m0 = tblk * TT * 32, rg = wave / KH;
    WideWave W;
    W.kh = wave % KH;
    W.r = lane & 31;
    W.j = lane >> 5;
    W.sb0 = ks * nsb / nks;
    W.n = (ks + 1) * nsb / nks - W.sb0;

    // groups past the last multiply the last one's rows (and store nothing)
    const int u = min(rb * kRG + rg, wide_groups(p) - 1);
    GemmSeg S = p.seg[0];
    int row0;  // the group's first row in its segment
    if (swi) {
        if (u & 1) S = p.seg[1];
        row0 = (u >> 1) * 32;
    } else {
#pragma unroll
        for (int i = 1; i < 4; i++)
            if (i < p.nseg && 2 * u >= p.seg[i].tile0) S = p.seg[i];
        row0 = (2 * u - S.tile0) * 16;
    }
    {
        const uint32_t tbb = (uint32_t)tile_block_bytes(S.fmt);
        W.w = make_rsrc(S.w, (uint32_t)(S.rows >> 4) * (uint32_t)nsb * tbb);
        W.wvo = (uint32_t)((row0 >> 4) + (W.r >> 4)) * (uint32_t)nsb * tbb;
    }
    // token tiles past the last read the last one (their products are dropped)
    const int last_tile = (p.M - 1) >> 5;
    W.x = make_rsrc(p.xp, (uint32_t)(last_tile + 1) * (uint32_t)nsb * kXTile);
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
        W.xtile[tt] = uni((uint32_t)min((m0 >> 5) + min(tt, TT - 1), last_tile) * (uint32_t)nsb * kXTile);

    // input norm (M <= 64, norm_parts <= 64)
    const bool has_norm = p.norm_ssq != nullptr;
    floatx16 acc[TT];
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[tt][i] = 0.f;
    switch (S.fmt) {
    case Q4_K: wide_body<Q4_K, TT, KH>(W, acc, wlds); break;
    case Q5_K: wide_body<Q5_K, TT, KH>(W, acc, wlds); break;
    case Q6_K: wide_body<Q6_K, TT, KH>(W, acc, wlds); break;
    default: wide_body<Q8_0, TT, KH>(W, acc, wlds); break;
    }

    // ---- the sums go through LDS, two token tiles at a time, as [wave][token
    // tile][token][row]: the chunk halves are added where they are read, and
    // outputs leave in runs of 128 bytes per token ----
    __shared__ float s_inv[64];
    if (has_norm) {
#pragma unroll
        for (int t = tid; t < 512; t += NT) {
            float nrm = 0.f;
            const int m = min(t >> 3, p.M - 1);
            for (int q = t & 7; q < p.norm_parts; q += 8) nrm += p.norm_ssq[m * p.norm_parts + q];
            nrm += __shfl_xor(nrm, 1);
            nrm += __shfl_xor(nrm, 2);
            nrm += __shfl_xor(nrm, 4);
            if ((t & 7) == 0) s_inv[t >> 3] = 1.0f / sqrtf(nrm / (float)p.K + p.norm_eps);
        }
    }
    constexpr int TR = TT < 2 ? 1 : 2;  // token tiles of a round
    float *Y = (float *)wlds;
    const int R = p.ntiles * 16, ngr = wide_groups(p);
#pragma unroll
    for (int t0 = 0; t0 < TT; t0 += TR) {
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < TR; tt++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(floatx4 *)(Y + (wave * TR + tt) * kYTile + W.r * kYPitch + 8 * q + 4 * W.j) =
                    floatx4{acc[t0 + tt][4 * q], acc[t0 + tt][4 * q + 1], acc[t0 + tt][4 * q + 2], acc[t0 + tt][4 * q + 3]};
        __syncthreads();
        // rows 4 c .. 4 c + 3 of group g for token tk of the round
        auto sum = [&](int g, int tk, int c) {
            const float *y = Y + (KH * g * TR + (tk >> 5)) * kYTile + (tk & 31) * kYPitch + 4 * c;
            floatx4 v = *(const floatx4 *)y;
            if constexpr (KH == 2) v += *(const floatx4 *)(y + TR * kYTile);
            return v;
        };
        if (swi) {
            // a thread: token tk, rows 4 c .. of both feature groups -> slots 0..7 of chunk c
            const int tk = tid % (32 * TR);
            const int m = m0 + t0 * 32 + tk, f0 = rb * 64;
            const float inv = has_norm ? s_inv[min(m, 63)] : 1.f;
#pragma unroll
            for (int c = tid / (32 * TR); c < 8; c += NT / (32 * TR)) {
                uint32_t o[4];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const floatx4 g = sum(2 * h, tk, c) * inv, v = sum(2 * h + 1, tk, c) * inv;
                    float a[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) a[i] = silu_w(g[i]) * v[i];
                    o[2 * h] = (uint32_t)f2h(a[0]) | ((uint32_t)f2h(a[2]) << 16);
                    o[2 * h + 1] = (uint32_t)f2h(a[1]) | ((uint32_t)f2h(a[3]) << 16);
                }
                if (m < p.M)
                    *(uintx4 *)(p.act + xt_index(m, frag_index(f0 + 4 * c), p.act_ld)) = uintx4{o[0], o[1], o[2], o[3]};
            }
            continue;
        }
        // a thread: rows 4 c .. of one token, the groups in turn; the NT / 8
        // tokens at a time are half a round, the round, or the round with the
        // groups halved
        constexpr int TP = NT / 8, GS = TP > 32 * TR ? 2 : 1, GN = kRG / GS;
#pragma unroll
        for (int tp = 0; tp < 32 * TR; tp += TP) {
            const int c = lane & 7, tk = tp + ((tid >> 3) & (32 * TR - 1)), ga = GS == 2 ? (wave >> 2) * GN : 0;
            const int m = m0 + t0 * 32 + tk;
            const bool in = m < p.M;
            const float inv = has_norm && nks == 1 ? s_inv[min(m, 63)] : 1.f;
            float bv = -INFINITY;
            int bi = 0x7fffffff;
#pragma unroll
            for (int g = ga; g < ga + GN; g++) {
                const int gu = rb * kRG + g;
                if (!in || gu >= ngr) continue;
                floatx4 y = sum(g, tk, c);
                const int n0 = gu * 32 + 4 * c;  // among the launch's rows
                if (nks > 1) {
                    // K slices: partial sums [ks][M][R]; the consumer of the output adds them in slice order
                    *(floatx4 *)(p.part + ((int64_t)ks * p.M + m) * R + n0) = y;
                    continue;
                }
                GemmSeg T = p.seg[0];
#pragma unroll
                for (int i = 1; i < 4; i++)
                    if (i < p.nseg && 2 * gu >= p.seg[i].tile0) T = p.seg[i];
                const int n1 = n0 - T.tile0 * 16;  // in the segment
                if (has_norm) y *= inv;
                float *o = T.out + (int64_t)m * T.ldo + T.col0 + n1;
                if (p.mode == GM_RESID) y += *(const floatx4u *)o;
                else if (T.bias) y += *(const floatx4 *)(T.bias + n1);
                *(floatx4u *)o = y;
                if (p.mode == GM_LOGITS) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int idx = T.col0 + n1 + i;
                        if (y[i] > -INFINITY && (y[i] > bv || (y[i] == bv && idx < bi))) {
                            bv = y[i];
                            bi = idx;
                        }
                    }
                }
            }
            if (p.mode == GM_LOGITS) {
#pragma unroll
                for (int o = 1; o < 8; o <<= 1) amax_merge(bv, bi, __shfl_xor(bv, o), __shfl_xor(bi, o));
                if (c == 0 && in) {
                    const int slot = GS == 2 ? rb * 2 + (wave >> 2) : rb;
                    p.amax_v[(int64_t)m * p.amax_ld + slot] = bv;
                    p.amax_i[(int64_t)m * p.amax_ld + slot] = bi;
                }
            }
        }
    }
}

// --------------------------------------------------------------------------
// Launch policy
// --------------------------------------------------------------------------
static int row_blocks(const GemmParams &p) { return (wide_groups(p) + kRG - 1) / kRG; }
static int token_blocks(int M, int tt) { return (M + 32 * tt - 1) / (32 * tt); }
static bool may_split(const GemmParams &p) { return p.allow_split && (p.mode == GM_STORE || p.mode == GM_RESID); }
// Token tiles of a workgroup: as few as hold the rows, at most four.  Above 64
// rows a launch of at most 64 workgroups, K slices included, takes two: most
// CUs are idle, and half the tiles shorten the chain that bounds it (512 wide,
// 1536 ffn, 96 rows: Q/K/V 8.3 -> 6.5 us, wo 7.6 -> 5.8, gate/up 9.4 -> 7.1,
// down 8.0 -> 5.9).  Larger launches lose: each weight is dequantised twice
// (14336 -> 4096 at 96 rows 21.3 -> 22.7).
static int wide_tt(const GemmParams &p) {
    if (p.M <= 32) return 1;
    if (p.M <= 64) return 2;
    return row_blocks(p) * token_blocks(p.M, 4) * (may_split(p) ? std::min(8, p.K / 256) : 1) <= 64 ? 2 : 4;
}
static int workgroups(const GemmParams &p) { return row_blocks(p) * token_blocks(p.M, wide_tt(p)); }
// Waves of a row group.  With two token tiles and more than one workgroup per
// CU to run, one: its four-wave workgroups sit two to a CU, where the eight-wave
// ones run in rounds whose prologue and epilogue nothing covers.  At 60 rows
// of 128256 x 4096 Q4_K (1002 workgroups) 97 us against 105, of gate/up 2 x 18944
// x 3584 Q8_0 (296) 46 against 49; where every workgroup has a CU of its own two
// are faster (2 x 14336 x 4096, 224 workgroups: 26.4 against 28.1).
static int wide_kh(const GemmParams &p) { return wide_tt(p) == 2 && workgroups(p) > 256 ? 1 : 2; }
// K slices, where the consumer of the output adds them.  Up to 64 rows the
// fewest with which no slice is longer than with the most that run at once, one
// workgroup to a CU: a 257th starts a second round (4608 x 3584 at 60 rows: 8
// slices, 288 workgroups 16.5 us, 7 slices 11.3).  Above, the count with the
// least modelled time: rounds of 256 workgroups at 6 us plus 1.9 us a
// superblock, and the partial sums written and read at 4 TB/s.  280 workgroups
// (3584 rows, 1251 tokens) take two rounds unsplit.  The weights are those that
// chose best, not a launch's own: full rounds measured 9.3 us plus 1.5 (Q4_K)
// to 1.67 us (Q8_0), but with 9.3 and 1.6 the rule took 1 slice for 4 (600 rows
// of 18944 -> 3584: 131 against 119 us, that prompt 2016 against 1971) and won
// nowhere above 64 rows by more than the runs differ.
int qwide_slices(const GemmParams &p) {
    if (!may_split(p)) return 1;
    const int wgs = workgroups(p), nsb = p.K / 256;
    const int64_t R = 16LL * p.ntiles;
    auto fits = [&](int ks) { return ks <= 8 && ks <= nsb && (ks == 1 || ks * p.M * R <= p.part_cap); };
    if (p.M <= 64) {
        int ks = 1;
        while (fits(ks + 1) && wgs * (ks + 1) <= 256) ks++;
        const int longest = (nsb + ks - 1) / ks;
        return (nsb + longest - 1) / longest;
    }
    int best = 1;
    double least = 0.0;
    for (int ks = 1; fits(ks); ks *= 2) {
        const int rounds = (wgs * ks + 255) / 256;
        const double us = rounds * (6.0 + 1.9 * nsb / ks) + (ks > 1 ? ks * p.M * R * 8.0 / 4e6 : 0.0);
        if (ks == 1 || us < least) {
            least = us;
            best = ks;
        }
    }
    return best;
}
int qwide_slots(const GemmParams &p) { return row_blocks(p) * (wide_tt(p) == 1 ? 2 : 1); }

template <int TT, int KH, int WPE>
static void wide_launch(const GemmParams &p, hipStream_t st, const LaunchTiming &tm) {
    const int nrb = row_blocks(p), nks = qwide_slices(p), ntb = token_blocks(p.M, TT);
    const size_t lds = wide_lds<TT, KH>();
    const WideArgs args{p, nrb, nks, ntb};
    const dim3 grid((unsigned)((nrb * nks + 7) / 8 * 8 * ntb)), block(wide_threads(KH));
    if (lds + sizeof(float) * 64 > 65536) {  // with s_inv
        static std::atomic<uint64_t> done{0};  // bit per device
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) throw BackendError("qwide: hipGetDevice");
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done.load(std::memory_order_acquire) & bit) || dev > 63) {
            if (hipFuncSetAttribute((const void *)k_qwide<TT, KH, WPE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds) != hipSuccess)
                throw BackendError("qwide: LDS size");
            done.fetch_or(bit, std::memory_order_release);
        }
    }
    if (tm.start && tm.stop)
        hipExtLaunchKernelGGL((k_qwide<TT, KH, WPE>), grid, block, lds, st, tm.start, tm.stop, 0, args);
    else hipLaunchKernelGGL((k_qwide<TT, KH, WPE>), grid, block, lds, st, args);
}

void launch_qwide(const GemmParams &p, hipStream_t st, const LaunchTiming &tm) {
    if (qwide_slices(p) > 1 && !p.part) throw BackendError("qgemm: split-K workspace missing");
    for (int i = 0; i < p.nseg; i++)
        if (p.seg[i].rows % 32 || p.seg[i].tile0 % 2) throw BackendError("qgemm: 32-row tiles above 16 tokens");
    const int tt = wide_tt(p);
    if (tt == 1) wide_launch<1, 2, 4>(p, st, tm);
    else if (tt == 4) wide_launch<4, 2, 2>(p, st, tm);
    else if (wide_kh(p) == 2) wide_launch<2, 2, 2>(p, st, tm);
    else wide_launch<2, 1, 2>(p, st, tm);
}

}  // namespace sd
