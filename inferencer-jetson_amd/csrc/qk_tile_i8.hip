// qk_tile_i8.hip - the INT8 multi-token product of many tokens on the fp16
// matrix cores.
//
// The arithmetic is qk_skinny.hip's (gemv_batch_dp4a over per-32 quantized
// activations, inferencer.cu:678-699; the sub-block combines of
// dot_q4_block_dp4a / dot_q6_block_dp4a, 520-542, 613-643):
//   Q4_K: d * sum_s xscale_s (sc_s I_s) - dmin * sum_s m_s xscale_s S_s
//   Q6_K: d * sum_c xscale_c (scale_2c I_2c + scale_2c+1 I_2c+1)
// but the integer scales move into the weight operand: sc * q (0..945) and
// scale * (code - 32) are exact in fp16 (a Q6_K product beyond 2048 as its
// rounded value plus the exact residual, a second chain), int8 activation
// codes are, and a 32-column sum of their products stays within 2^24, so two
// (four) v_mfma_f32_32x32x16_f16 leave sc_s I_s as an exact fp32 integer.
// What remains per output and 32 columns is one fma by the activation scale,
// where int32 dots take a conversion, a product by the row's scale and an
// fma: that combine, not the matrix cores or memory, bounds the int32 form.
//
// Weights are the A operand (output register = weight row), tokens the B
// operand (output lane = token), so the activation scale is one value a lane.
// A workgroup of four waves takes 64 tokens and 128 rows, or 64 rows of gate
// and of up, a 32-row tile a wave; a decoded weight operand meets both token
// tiles.  The workgroup converts its tokens' codes to fp16 operands in LDS
// half a block (128 columns) at a time while the other half multiplies;
// weights are decoded in registers from raw bytes requested a half ahead.
// Three workgroups fit a CU; a block takes one alone 2.4 us and three 5.5 us,
// against 3.0 us of VALU work: what is left is the wait for weights and the
// barrier of each half.
//
// Sums: a Q4_K block's dots and mins are added to each other before they
// enter the running sum (1.55e-7 of float64 over 16 blocks, 1.6e-7 over 32;
// the int32 kernels 1.62 and 1.65e-7; with every min product entering the
// running sum on its own 2.0 and 2.2 to 3.3e-7), and sums of many blocks have
// two levels (kShortBlocks).
//
// Measured against the looping int32 kernel: a 3B feed-forward block (gate /
// up 8192 x 3072 Q4_K, down 3072 x 8192 Q6_K split) on 517 tokens 402 -> 226
// us, its down product alone 165 -> 97 us; Q4_K 8192 x 8192 on 1000 tokens 452
// -> 278 us.  Tried: two row tiles a wave (two waves a SIMD, spills: 298 us),
// no step of dots ahead of the combine (256 us), the mins on the bf16 matrix
// instructions in three exact parts (4 to 19 % more: the splitting), and two
// levels of sums at every length (2 to 5 % more).
#include "qk_operands.h"

#include <algorithm>

namespace qk {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kTok = 32, kRowTile = 32;
constexpr int kPairRows = 64, kStoreRows = 128;   // weight rows of a workgroup (of each matrix of a pair)
constexpr int kHalfTile = 8 * 1024;                // one token tile's half block: 4 sub-blocks x 2 operands x 1 KB
constexpr int kMaxSplits = 8;
constexpr int kMaxItems = 2048;   // workgroups of a split launch at most: bounds the sums to 64 MB

struct TiMatrix {
    const uint8_t *w;
    float *y;
    int rows, row_bytes, ldy;
    int group_begin;   // first workgroup row group
    int row_begin;     // first row in the split sums
    int vec;           // float4 access to y allowed
};

struct TiParams {
    TiMatrix mat[QK_MAX_FUSED];
    int n_mats, n_tokens, nb;
    const int8_t *xq;
    const float *xs;
    int ldxq, ldxs;
    int groups, tgroups, tiles;         // row groups, token groups, token tiles
    int splits, blocks_per_split;
    int accumulate;
    int part_rows;                      // rows of the split sums
    float *partials;                    // splits > 1: [split][token][part_rows]
    int8_t *out_xq;
    float *out_xs;
    int out_ldxq, out_ldxs;
};

// LDS: two halves' operands, their activation scales ([half][tile][sub-block]
// [token]), three halves' scale * sum products (the same; a block's two are read
// when it ends, while the next one's first are written: those of first halves
// alternate, slots 0 and 1, second halves take slot 2), then d of the waves' rows.
__host__ __device__ constexpr int ti_lds(int tt) {
    return 2 * tt * kHalfTile + (2 + 3) * tt * 4 * kTok * 4 + 4 * kRowTile * 4;
}

// A lane's 32-bit offset from a wave-uniform base, kept in that form: the
// compiler otherwise carries 64-bit lane pointers through the loop, spills
// some and waits for the weights in flight when it reloads them.
__device__ __forceinline__ uint32_t lane_offset(uint32_t lane, uint32_t uniform) {
    uint32_t o = lane + uniform;
    asm("" : "+v"(o));
    return o;
}

// Half h (sub-blocks 4h .. 4h + 3) of the lane's row, column half kh of each
// sub-block (columns 16 kh .. + 15).  Q4_K: qs of groups 2h, 2h + 1 (low and
// high nibbles: sub-blocks); Q6_K: the two ql runs and the qh run.
template <bool Q4>
struct RawI8 {
    uint4 q[Q4 ? 2 : 3];
};
template <int TYPE>
__device__ __forceinline__ RawI8<TYPE == QK_TYPE_Q4_K> load_half(const uint8_t *base, uint32_t ofs, int b, int nb,
                                                                    int kh, int h) {
    RawI8<TYPE == QK_TYPE_Q4_K> r;
    if constexpr (TYPE == QK_TYPE_Q4_K) {
        const uint32_t o = lane_offset(ofs + 16 * kh, b * 144);
        r.q[0] = load16(base + o + (16 + 64 * h));
        r.q[1] = load16(base + o + (48 + 64 * h));
    } else {
        const Q6Fields f = q6_fields(base, nb, b, TYPE == QK_TYPE_Q6_K_SPLIT);
        r.q[0] = load16(f.ql + 64 * h + (ofs + 16 * kh));
        r.q[1] = load16(f.ql + 64 * h + 32 + (ofs + 16 * kh));
        r.q[2] = load16(f.qh + 32 * h + (ofs + 16 * kh));
    }
    return r;
}

// Q4_K: the 16-byte header; Q6_K: the sixteen scales and d.
struct Header {
    uint4 v;
    uint32_t d;
};
template <int TYPE>
__device__ __forceinline__ Header load_header(const uint8_t *base, uint32_t ofs, int b, int nb) {
    if constexpr (TYPE == QK_TYPE_Q4_K) {
        return {load16(base + lane_offset(ofs, b * 144)), 0};
    } else {
        const Q6Fields f = q6_fields(base, nb, b, TYPE == QK_TYPE_Q6_K_SPLIT);
        return {load16(f.sc + ofs), load2(f.d + ofs)};
    }
}

// Sub-block s of the half as its two operands (words 2m, 2m + 1 of the run;
// a word's columns in the order 0, 2, 1, 3), scaled; wb: Q6_K residuals.
template <bool Q4>
__device__ __forceinline__ void decode(const RawI8<Q4> &r, int s, _Float16 sc, half8 (&w)[2], half8 (&wb)[2]) {
    #pragma unroll
    for (int m = 0; m < 2; ++m) {
        uint32_t a[4], e[4];
        #pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t v = quad_word(r.q[Q4 ? s >> 1 : s & 1], 2 * m + i);
            if constexpr (Q4) {
                const uint32_t mask = s & 1 ? 0x00F000F0u : 0x000F000Fu;
                const half2v f = h2(s & 1 ? sc * static_cast<_Float16>(0.0625f) : sc);
                const half2v o = h2(static_cast<_Float16>(s & 1 ? -64.f : -1024.f) * sc);
                a[2 * i] = as_u32(__builtin_elementwise_fma(as_h2((v & mask) | 0x64006400u), f, o));
                a[2 * i + 1] = as_u32(__builtin_elementwise_fma(as_h2(((v >> 8) & mask) | 0x64006400u), f, o));
            } else {
                const uint32_t hq = quad_word(r.q[2], 2 * m + i);
                const half2v f = h2(sc);
                if (s == 0) {
                    decode_q6_pair<0, 0>(v, hq, f, a[2 * i], e[2 * i]);
                    decode_q6_pair<8, 8>(v, hq, f, a[2 * i + 1], e[2 * i + 1]);
                } else if (s == 1) {
                    decode_q6_pair<0, 2>(v, hq, f, a[2 * i], e[2 * i]);
                    decode_q6_pair<8, 10>(v, hq, f, a[2 * i + 1], e[2 * i + 1]);
                } else if (s == 2) {
                    decode_q6_pair<4, 4>(v, hq, f, a[2 * i], e[2 * i]);
                    decode_q6_pair<12, 12>(v, hq, f, a[2 * i + 1], e[2 * i + 1]);
                } else {
                    decode_q6_pair<4, 6>(v, hq, f, a[2 * i], e[2 * i]);
                    decode_q6_pair<12, 14>(v, hq, f, a[2 * i + 1], e[2 * i + 1]);
                }
            }
        }
        w[m] = __builtin_bit_cast(half8, make_uint4(a[0], a[1], a[2], a[3]));
        if constexpr (!Q4) wb[m] = __builtin_bit_cast(half8, make_uint4(e[0], e[1], e[2], e[3]));
    }
}

// Four int8 codes as fp16 in the order 0, 2, 1, 3: 1024 + (code + 128) - 1152.
__device__ __forceinline__ uint2 codes_to_h(uint32_t v) {
    const uint32_t x = v ^ 0x80808080u;
    const half2v o = h2(static_cast<_Float16>(-1152.f));
    return make_uint2(as_u32(as_h2((x & 0x00FF00FFu) | 0x64006400u) + o),
                      as_u32(as_h2(((x >> 8) & 0x00FF00FFu) | 0x64006400u) + o));
}

// Blocks that one running sum takes in the short form: up to these, its error
// against 64 bits is not above the int32 kernels' (1.65e-7 at 32 Q4_K blocks in
// two sums of 16; 9.2e-8 for Q6_K, whose 16-block sums reach 9.7e-8).  The long
// form keeps a second level, every kRun blocks added to a total: 1.6e-7 and
// 9.4e-8 up to 96 blocks, at two workgroups a CU (registers).
template <int TYPE>
constexpr int kShortBlocks = TYPE == QK_TYPE_Q4_K ? 16 : 12;
constexpr int kRun = 8;

// One workgroup: TT token tiles from tile0 (all exist) x its rows x the
// blocks of a split.
template <int TYPE, int TT, bool PAIR, bool LONG>
__device__ __forceinline__ void tile_body(const TiParams &p, const TiMatrix &M, int row0, int tile0, int split,
                                          unsigned char *lds) {
    constexpr bool Q4 = TYPE == QK_TYPE_Q4_K;
    const int lane = threadIdx.x & 63, kh = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *const scales = reinterpret_cast<float *>(lds + 2 * TT * kHalfTile);   // [half][tile][4][32]
    constexpr int kPlane = TT * 4 * kTok;                                        // one half's
    float *const sums = scales + 2 * kPlane;                                     // [slot][tile][4][32], scale * sum of codes
    float *const drow = sums + 3 * kPlane + wave * kRowTile;                     // d of the wave's rows
    // Rows past the matrix read its last row (and store nothing).
    // A pair's waves 0, 1 take the gate rows, 2, 3 the same rows of up.  Lane
    // addresses: a wave-uniform base and a 32-bit offset.
    const TiMatrix &W = PAIR ? p.mat[wave >> 1] : M;
    const int r0 = row0 + (PAIR ? wave & 1 : wave) * kRowTile;
    const int first = min(r0, W.rows - 1);
    const uint8_t *const wbase = W.w + static_cast<size_t>(first) * W.row_bytes;
    const uint32_t wofs = static_cast<uint32_t>(min(r0 + col, W.rows - 1) - first) * W.row_bytes;
    const int64_t t0 = static_cast<int64_t>(tile0) * kTok;
    const int8_t *const xq = p.xq + t0 * p.ldxq + wave * 32;
    const float *const xs = p.xs + t0 * p.ldxs + wave;
    uint32_t tofs[TT];
    #pragma unroll
    for (int u = 0; u < TT; ++u) tofs[u] = static_cast<uint32_t>(min(u * kTok + col, p.n_tokens - 1 - tile0 * kTok));
    const int b0 = split * p.blocks_per_split, b1 = min(p.nb, b0 + p.blocks_per_split);

    // A wave converts sub-block `wave` of the half for every tile: the lane's
    // token (col) and column half.
    uint4 codes[TT];
    float cs[TT];
    auto request = [&](int b, int h) {
        #pragma unroll
        for (int u = 0; u < TT; ++u) {
            codes[u] = *reinterpret_cast<const uint4 *>(xq + b * 256 + h * 128 + (tofs[u] * static_cast<uint32_t>(p.ldxq) + kh * 16));
            cs[u] = (xs + b * 8 + h * 4)[tofs[u] * static_cast<uint32_t>(p.ldxs)];
        }
    };
    auto commit = [&](int block, int h) {
        #pragma unroll
        for (int u = 0; u < TT; ++u) {
            unsigned char *dst = lds + (h * TT + u) * kHalfTile + wave * 2048 + lane * 16;
            const uint2 a = codes_to_h(codes[u].x), b = codes_to_h(codes[u].y);
            const uint2 c = codes_to_h(codes[u].z), d = codes_to_h(codes[u].w);
            *reinterpret_cast<uint4 *>(dst) = make_uint4(a.x, a.y, b.x, b.y);
            *reinterpret_cast<uint4 *>(dst + 1024) = make_uint4(c.x, c.y, d.x, d.y);
            // (Both column halves write the same values.)
            float *const at = scales + wave * kTok + col + u * 4 * kTok;
            at[h * kPlane] = cs[u];
            if constexpr (Q4) {
                int sum = __builtin_amdgcn_sdot4(static_cast<int>(codes[u].x), 0x01010101, 0, false);
                sum = __builtin_amdgcn_sdot4(static_cast<int>(codes[u].y), 0x01010101, sum, false);
                sum = __builtin_amdgcn_sdot4(static_cast<int>(codes[u].z), 0x01010101, sum, false);
                sum = __builtin_amdgcn_sdot4(static_cast<int>(codes[u].w), 0x01010101, sum, false);
                sum += __shfl_xor(sum, 32);
                at[(2 + (h ? 2 : block & 1)) * kPlane] = static_cast<float>(sum) * cs[u];
            }
        }
    };

    float16v zero;
    #pragma unroll
    for (int k = 0; k < 16; ++k) zero[k] = 0.f;
    float16v acc[TT], blk[TT];
    #pragma unroll
    for (int u = 0; u < TT; ++u) acc[u] = blk[u] = zero;
    float16v total[LONG ? TT : 1];
    if constexpr (LONG)
        #pragma unroll
        for (int u = 0; u < TT; ++u) total[u] = zero;

    request(b0, 0);
    Header hdr = load_header<TYPE>(wbase, wofs, b0, p.nb);
    RawI8<Q4> cur = load_half<TYPE>(wbase, wofs, b0, p.nb, kh, 0);
    commit(b0, 0);
    __syncthreads();
    for (int b = b0; b < b1; ++b) {
        const int bn = min(b + 1, b1 - 1);   // the last block requests itself again (in bounds)
        Header hdr_next = hdr;
        uint32_t mn4[2];   // Q4_K: the halves' mins
        #pragma unroll
        for (int h = 0; h < 2; ++h) {
            const RawI8<Q4> next = load_half<TYPE>(wbase, wofs, h ? bn : b, p.nb, kh, h ^ 1);
            if (h) hdr_next = load_header<TYPE>(wbase, wofs, bn, p.nb);
            __builtin_amdgcn_sched_barrier(0);
            uint32_t sc4;   // Q4_K: the half's scales; Q6_K: column half kh's
            if constexpr (Q4) {
                q4k_scale_min4(hdr.v, h, sc4, mn4[h]);
            } else {
                const uint32_t lo = h ? hdr.v.z : hdr.v.x, hi = h ? hdr.v.w : hdr.v.y;
                sc4 = __builtin_amdgcn_perm(hi, lo, kh ? 0x07050301u : 0x06040200u);
            }
            if (h == 0) drow[col] = f16_bits_to_f32(Q4 ? hdr.v.x & 0xFFFFu : hdr.d);
            const unsigned char *op = lds + h * TT * kHalfTile + lane * 16;
            const float *sx = scales + h * kPlane + col;
            // Each Q4_K step issues one tile's dots, then combines the step
            // before's; Q6_K has the registers for one tile's only.
            half8 w[2], wb[2];
            float16v tp = zero;
            float fp = 0.f;
            auto combine = [&](int j, const float16v &v, float scale) {
                #pragma unroll
                for (int k = 0; k < 16; ++k)
                    blk[j % TT][k] = h == 0 && j < TT ? v[k] * scale : fmaf(v[k], scale, blk[j % TT][k]);
            };
            #pragma unroll
            for (int i = 0; i < 4 * TT; ++i) {
                const int s = i / TT, u = i % TT;
                if (i == 2 * TT) request(h ? bn : b, h ^ 1);   // later than the weights: registers
                if (u == 0) decode<Q4>(cur, s, Q4 ? u8_to_h(sc4 >> (8 * s)) : s8_to_h(sc4 >> (8 * s)), w, wb);
                const half8 x0 = *reinterpret_cast<const half8 *>(op + u * kHalfTile + s * 2048);
                const half8 x1 = *reinterpret_cast<const half8 *>(op + u * kHalfTile + s * 2048 + 1024);
                const float f = sx[(u * 4 + s) * kTok];
                float16v t = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[0], x0, zero, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[1], x1, t, 0, 0, 0);
                if constexpr (!Q4) {
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[0], x0, t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[1], x1, t, 0, 0, 0);
                }
                if constexpr (Q4) {
                    if (i > 0) combine(i - 1, tp, fp);
                    tp = t;
                    fp = f;
                    if (i == 4 * TT - 1) combine(i, tp, fp);
                } else {
                    combine(i, t, f);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (h == 1) {
                // Both halves' sums are still in LDS; dmin m of the lane's row,
                // sub-blocks 2 j + kh.
                float am[4];
                const float *const sl = sums + (b & 1) * kPlane + lane, *const sh = sums + 2 * kPlane + lane;
                if constexpr (Q4) {
                    const float dmin = -f16_bits_to_f32(hdr.v.x >> 16);
                    #pragma unroll
                    for (int j = 0; j < 4; ++j)
                        am[j] = dmin * static_cast<float>((mn4[j >> 1] >> (16 * (j & 1) + 8 * kh)) & 0xFFu);
                }
                float d[16];
                #pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = *reinterpret_cast<const float4 *>(drow + 8 * q + 4 * kh);
                    d[4 * q] = v.x;
                    d[4 * q + 1] = v.y;
                    d[4 * q + 2] = v.z;
                    d[4 * q + 3] = v.w;
                }
                // The block's mins -- the fp32 product of dmin m and scale *
                // sum over its eight sub-blocks -- and its dots meet first:
                // each is about twice their sum, so the running sum takes
                // one rounding a block, of the block's own size.
                float16v tm[TT];
                if constexpr (Q4) {
                    #pragma unroll
                    for (int j = 0; j < 4; ++j)
                        #pragma unroll
                        for (int u = 0; u < TT; ++u)
                            tm[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                am[j], (j >> 1 ? sh : sl)[(u * 4 + 2 * (j & 1)) * kTok], j ? tm[u] : zero, 0, 0, 0);
                }
                #pragma unroll
                for (int u = 0; u < TT; ++u)
                    #pragma unroll
                    for (int k = 0; k < 16; ++k)
                        acc[u][k] = Q4 ? acc[u][k] + fmaf(d[k], blk[u][k], tm[u][k]) : fmaf(d[k], blk[u][k], acc[u][k]);
            }
            commit(h ? b + 1 : b, h ^ 1);
            __syncthreads();
            cur = next;
        }
        hdr = hdr_next;
        if constexpr (LONG) {
            const bool ends = b + 1 == b1;
            if ((b - b0) % kRun == kRun - 1 || ends) {
                #pragma unroll
                for (int u = 0; u < TT; ++u) {
                    total[u] += acc[u];
                    acc[u] = ends ? total[u] : zero;
                }
            }
        }
    }

    if constexpr (PAIR) {
        // The up waves hand their sums to the gate waves through the operand
        // area, free since the last barrier ([wave][tile][register][lane]).
        float *const x = reinterpret_cast<float *>(lds) + (wave & 1) * TT * 1024 + lane;
        if (wave >= 2) {
            #pragma unroll
            for (int u = 0; u < TT; ++u)
                #pragma unroll
                for (int k = 0; k < 16; ++k) x[u * 1024 + k * 64] = acc[u][k];
        }
        __syncthreads();
        if (wave >= 2) return;
        #pragma unroll
        for (int u = 0; u < TT; ++u)
            #pragma unroll
            for (int k = 0; k < 16; ++k) blk[u][k] = x[u * 1024 + k * 64];
    }

    // Register k holds row 8 * (k / 4) + 4 * kh + k % 4 of its tile, the lane
    // token col.
    #pragma unroll
    for (int u = 0; u < TT; ++u) {
        const int t = (tile0 + u) * kTok + col;
        if constexpr (PAIR) {
            // A token's 32 outputs of the tile are one quantization group:
            // two lanes, sixteen values each (quantize_group_store's rule).
            if (r0 >= M.rows) continue;
            float v[16], amax = 0.f;
            #pragma unroll
            for (int k = 0; k < 16; ++k) {
                v[k] = silu_mul_value(acc[u][k], blk[u][k]);
                amax = fmaxf(amax, fabsf(v[k]));
            }
            amax = fmaxf(amax, __shfl_xor(amax, 32));
            const float scale = amax > 0.f ? amax / 127.f : 1.f;
            if (t >= p.n_tokens) continue;
            if (kh == 0) p.out_xs[static_cast<int64_t>(t) * p.out_ldxs + r0 / 32] = scale;
            #pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t word = 0;
                #pragma unroll
                for (int k = 0; k < 4; ++k) {
                    int c = static_cast<int>(rintf(v[4 * q + k] / scale));
                    c = c < -127 ? -127 : (c > 127 ? 127 : c);
                    word |= (static_cast<uint32_t>(c) & 0xFFu) << (8 * k);
                }
                *reinterpret_cast<uint32_t *>(p.out_xq + static_cast<int64_t>(t) * p.out_ldxq + r0 + 8 * q + 4 * kh) = word;
            }
        } else {
            if (t >= p.n_tokens) continue;
            if (r0 >= M.rows) continue;
            #pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + 8 * q + 4 * kh;
                float4 v = make_float4(acc[u][4 * q], acc[u][4 * q + 1], acc[u][4 * q + 2], acc[u][4 * q + 3]);
                if (p.partials) {
                    *reinterpret_cast<float4 *>(p.partials + (static_cast<size_t>(split) * p.n_tokens + t) * p.part_rows +
                                                M.row_begin + r) = v;
                    continue;
                }
                float *y = M.y + static_cast<int64_t>(t) * M.ldy + r;
                if (M.vec) {   // rows a multiple of 4: all four or none
                    if (r < M.rows) {
                        if (p.accumulate) {
                            const float4 o = *reinterpret_cast<const float4 *>(y);
                            v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
                        }
                        *reinterpret_cast<float4 *>(y) = v;
                    }
                } else {
                    const float e[4] = {v.x, v.y, v.z, v.w};
                    #pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (r + k < M.rows) y[k] = p.accumulate ? e[k] + y[k] : e[k];
                }
            }
        }
    }
}

// In xcd_item's list the token groups of one row group are neighbours: they share
// its weight bytes.
template <int TYPE, bool PAIR, bool LONG>
__global__ __launch_bounds__(256, LONG ? 2 : 3) void tile_i8(TiParams p) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int item = xcd_item(static_cast<int>(blockIdx.x), p.groups * p.tgroups * p.splits);
    if (item < 0) return;
    const int tgroup = item % p.tgroups, rest = item / p.tgroups;
    const int split = rest % p.splits, group = rest / p.splits;
    int m = 0;
    if constexpr (!PAIR) {
        #pragma unroll
        for (int i = 1; i < QK_MAX_FUSED; ++i) m += (i < p.n_mats && group >= p.mat[i].group_begin) ? 1 : 0;
        m = __builtin_amdgcn_readfirstlane(m);
    }
    const TiMatrix &M = p.mat[m];
    const int row0 = (group - M.group_begin) * (PAIR ? kPairRows : kStoreRows), tile0 = tgroup * 2;
    // A ragged last group of one tile does the work of one.
    if (tile0 + 1 < p.tiles)
        tile_body<TYPE, 2, PAIR, LONG>(p, M, row0, tile0, split, lds);
    else
        tile_body<TYPE, 1, PAIR, LONG>(p, M, row0, tile0, split, lds);
}

// Adds the splits' sums in split order and stores: four rows of one token a
// thread.
__global__ __launch_bounds__(256) void tile_i8_reduce(TiParams p) {
    const int quads = p.part_rows / 4;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= static_cast<int64_t>(quads) * p.n_tokens) return;
    const int t = static_cast<int>(i / quads), pr = static_cast<int>(i % quads) * 4;
    const float *src = p.partials + static_cast<size_t>(t) * p.part_rows + pr;
    const size_t stride = static_cast<size_t>(p.n_tokens) * p.part_rows;
    float4 v[kMaxSplits];
    #pragma unroll
    for (int s = 0; s < kMaxSplits; ++s)
        if (s < p.splits) v[s] = *reinterpret_cast<const float4 *>(src + s * stride);
    float4 a = v[0];
    #pragma unroll
    for (int s = 1; s < kMaxSplits; ++s)
        if (s < p.splits) a = make_float4(a.x + v[s].x, a.y + v[s].y, a.z + v[s].z, a.w + v[s].w);
    int m = 0;
    #pragma unroll
    for (int j = 1; j < QK_MAX_FUSED; ++j) m += (j < p.n_mats && pr >= p.mat[j].row_begin) ? 1 : 0;
    const TiMatrix &M = p.mat[m];
    const int r = pr - M.row_begin;
    const float e[4] = {a.x, a.y, a.z, a.w};
    float *y = M.y + static_cast<int64_t>(t) * M.ldy + r;
    #pragma unroll
    for (int k = 0; k < 4; ++k)
        if (r + k < M.rows) y[k] = p.accumulate ? e[k] + y[k] : e[k];
}

template <int TYPE, bool PAIR>
void launch_type(const TiParams &p, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((p.groups * p.tgroups * p.splits + 7) / 8 * 8));
    const size_t lds = ti_lds(std::min(p.tiles, 2));
    if (p.blocks_per_split > kShortBlocks<TYPE>)
        hipLaunchKernelGGL((tile_i8<TYPE, PAIR, true>), grid, dim3(256), lds, stream, p);
    else
        hipLaunchKernelGGL((tile_i8<TYPE, PAIR, false>), grid, dim3(256), lds, stream, p);
}

template <bool PAIR>
void launch(int type, const TiParams &p, hipStream_t stream) {
    if (type == QK_TYPE_Q4_K)
        launch_type<QK_TYPE_Q4_K, PAIR>(p, stream);
    else if (type == QK_TYPE_Q6_K)
        launch_type<QK_TYPE_Q6_K, PAIR>(p, stream);
    else
        launch_type<QK_TYPE_Q6_K_SPLIT, PAIR>(p, stream);
}

}  // namespace

// Without a pair, few tokens leave part of a token group empty and the sum
// traffic outweighs the gain: Q4_K 8192 x 3072 takes 33 / 41 us here and 26 /
// 37 there on 96 / 130 tokens, 46 and 51 on 256; Q6_K 40 and 36 on 96, 49 and
// 50 on 130; rows of 14336 gain from 40 tokens on (38 and 56).
static int least_tokens(bool q4, int nb) { return q4 ? 192 : nb > 32 ? 0 : 128; }

// Splits of least modelled time: a block takes a workgroup kBlockUs[r] with r
// workgroups on its CU (measured, Q4_K), split sums their traffic and a
// launch.  A pair is not split: its epilogue needs whole sums.  Launches of
// fewer workgroups than CUs stay with launch_skinny_i8's kernels (gate / up
// 8192 x 3072, 64 tokens: 128 workgroups, 41 us against 34).
int tile_i8_splits(const qk_matrix *mats, int n_mats, int cols, int n_tokens, int ldxq, int ldscale, bool pair,
                   size_t workspace_size) {
    // A 64-token tile's offsets are 32 bits.
    if (ldxq >= 1 << 26 || ldscale >= 1 << 24) return 0;
    const int nb = cols / 256, cus = std::max(1, device_info().cus);
    const bool q4 = mats[0].type == QK_TYPE_Q4_K;
    if (!pair && n_tokens < least_tokens(q4, nb)) return 0;
    int groups = 0;
    size_t part_rows = 0;
    for (int i = 0; i < (pair ? 1 : n_mats); ++i) {
        groups += (mats[i].rows + (pair ? kPairRows : kStoreRows) - 1) / (pair ? kPairRows : kStoreRows);
        part_rows += (mats[i].rows + kRowTile - 1) / kRowTile * kRowTile;
    }
    const int64_t items = static_cast<int64_t>(groups) * ((n_tokens + 2 * kTok - 1) / (2 * kTok));
    if (items * kMaxSplits > (1 << 30)) return 0;
    constexpr double kBlockUs[3] = {2.4, 3.8, 5.5}, kReduceUs = 4., kSumUsPerMb = 0.4;
    const size_t bytes = part_rows * n_tokens * sizeof(float);
    const double mb = 1e-6 * static_cast<double>(bytes);
    auto least_of = [&](int max_splits) {
        int best = 0;
        double least = 0;
        for (int s = 1; s <= max_splits; ++s) {
            if (items * s < cus || (s > 1 && items * s > kMaxItems)) continue;
            const int per = (nb + s - 1) / s;
            const int resident = per > (q4 ? kShortBlocks<QK_TYPE_Q4_K> : kShortBlocks<QK_TYPE_Q6_K>) ? 2 : 3;
            const int64_t wgs = items * s, full = wgs / (resident * cus), rest = wgs % (resident * cus);
            const double us = per * (full * kBlockUs[resident - 1] + (rest ? kBlockUs[(rest - 1) / cus] : 0.)) +
                              (s > 1 ? kReduceUs + kSumUsPerMb * mb * s : 0.);
            if (!best || us < least) {
                best = s;
                least = us;
            }
        }
        return best;
    };
    const int best = least_of(pair ? 1 : std::min(nb, kMaxSplits));
    // Less than the queried size: the splits that fit.
    return best > 1 && best * bytes > workspace_size ? least_of(static_cast<int>(workspace_size / bytes)) : best;
}

// Bytes that tile_i8_splits' choice takes, for any types and any division of
// `tiles` 32-row tiles over matrices, at this token count and below: splits *
// tokens is at most kMaxSplits times them, and kMaxItems workgroups' tokens.
size_t tile_i8_workspace_bytes(int cols, int tiles, int n_tokens) {
    const int nb = cols / 256;
    if (n_tokens < std::min(least_tokens(true, nb), least_tokens(false, nb))) return 0;
    const int64_t groups = (static_cast<int64_t>(tiles) * kRowTile + kStoreRows - 1) / kStoreRows;
    const int64_t split_tokens = std::min<int64_t>(static_cast<int64_t>(std::min(nb, kMaxSplits)) * n_tokens,
                                                   kMaxItems / std::max<int64_t>(1, groups - QK_MAX_FUSED) * 2 * kTok);
    return static_cast<size_t>(split_tokens) * tiles * kRowTile * sizeof(float);
}

int launch_tile_i8(int splits, const qk_matrix *mats, int n_mats, const int *ldy, const int8_t *xq, int ldxq,
                   const float *xscale, int ldscale, int cols, int n_tokens, int accumulate, int8_t *out_xq,
                   float *out_xs, int out_ldxq, int out_ldxs, void *workspace, hipStream_t stream, const char *where) {
    TiParams p{};
    const bool pair = out_xq != nullptr;
    p.n_mats = n_mats;
    p.n_tokens = n_tokens;
    p.nb = cols / 256;
    p.xq = xq;
    p.xs = xscale;
    p.ldxq = ldxq;
    p.ldxs = ldscale;
    p.accumulate = accumulate;
    p.out_xq = out_xq;
    p.out_xs = out_xs;
    p.out_ldxq = out_ldxq;
    p.out_ldxs = out_ldxs;
    for (int i = 0; i < n_mats; ++i) {
        TiMatrix &M = p.mat[i];
        M.w = static_cast<const uint8_t *>(mats[i].w);
        M.y = mats[i].y;
        M.rows = mats[i].rows;
        M.row_bytes = static_cast<int>(row_bytes(mats[i].type, p.nb));
        M.ldy = ldy ? ldy[i] : mats[i].rows;
        M.group_begin = pair ? 0 : p.groups;
        M.row_begin = p.part_rows;
        M.vec = M.rows % 4 == 0 && M.ldy % 4 == 0 && aligned(M.y, 16);
        if (!pair || i == 0) p.groups += pair ? (M.rows + kPairRows - 1) / kPairRows : (M.rows + kStoreRows - 1) / kStoreRows;
        p.part_rows += (M.rows + kRowTile - 1) / kRowTile * kRowTile;
    }
    p.tiles = (n_tokens + kTok - 1) / kTok;
    p.tgroups = (p.tiles + 1) / 2;
    p.blocks_per_split = (p.nb + splits - 1) / splits;
    p.splits = (p.nb + p.blocks_per_split - 1) / p.blocks_per_split;   // none empty
    if (p.splits > 1) p.partials = static_cast<float *>(workspace);
    if (pair)
        launch<true>(mats[0].type, p, stream);
    else
        launch<false>(mats[0].type, p, stream);
    if (p.splits > 1) {
        const int64_t quads = static_cast<int64_t>(p.part_rows) / 4 * n_tokens;
        hipLaunchKernelGGL(tile_i8_reduce, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, stream, p);
    }
    return launch_status(where);
}

}  // namespace qk
