// qk_few.hip - products of 2 to 7 tokens with enough weights for it (few_pays): a
// few sequences decoding together, a few speculated tokens.
//
// One GEMV column per token decodes every weight once per token (their
// re-reads come from cache).  Here every weight is read and decoded once, into
// an MFMA operand for all of them: the 16 rows of v_mfma_f32_16x16x32_f16's
// other operand are eight token slots' fp16 high halves and their low halves,
// so one chain gives both parts of the 22-bit activations (csrc/qk_batched.
// hip's arithmetic).
//
//   * Wave w of a workgroup owns block w of the rows (two blocks each from 17
//     to 32): its activations stay in 32 registers a block, converted from
//     fp32 x by every workgroup (one coalesced read a token, through the
//     wave's own LDS into operand order), so the call needs no workspace and
//     no launch before it.
//   * The workgroup walks 16-row tiles (two at a time where there are enough,
//     or a gate and an up tile): a lane loads one row's quarter block, eight
//     16-byte operands, with the next tiles' bytes in flight.  The waves' sums
//     meet in LDS in wave order, one barrier a step.
//   * With `pair` the epilogue forms SiLU(gate) * up.
//
// Bound by the conversion (0.5 to 0.8 us a token) and the waves' meetings up to
// some 20 MB, then by the decode: 0.22 us a MB of Q4_K (4.5 TB/s) and 0.29 of
// split Q6_K (3.4), where the one-token GEMV streams 5.2 and 5.6.  Measured
// against the GEMV columns at 4 and 7 tokens: Q4_K 128256 x 2048 80.7 -> 38.1 and
// 148 -> 40.8 us, split Q6_K 118 -> 65 and 210 -> 64 us, Q4_K 16384 x 3072 21.5
// -> 13.6 and 34.8 -> 16.1 us; the 3B feed-forward block of 4 tokens 50.2 -> 34.7
// us.  (Converting in the operand's own lanes, 16-byte reads 256 bytes apart,
// took 3 to 8 us more.)
#include "qk_internal.h"
#include "qk_operands.h"
#include "qk_records.h"

#include <algorithm>

namespace qk {
namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kSlots = 8;            // token slots of an operand; a launch takes up to kSlots - 1 tokens
constexpr int kTileRows = 16;
constexpr int kMaxWaves = 16;

struct FewMatrix {
    const uint8_t *w;
    float *y;
    int rows, type, ldy;
    int64_t row_bytes;
    int block_begin, blocks;   // the matrix's workgroups
};

struct FewParams {
    FewMatrix mat[QK_MAX_FUSED];
    int n_mats;
    const float *x;
    int ldx, n_tokens, nb;
    const float *norm_w;   // x enters as RMSNorm(x) * norm_w
    float norm_eps;
    const float *up;       // x enters as SiLU(x) * up (up has x's layout)
    int accumulate;        // y += W x
    int pair;              // y0 = SiLU(W0 x) * (W1 x)
};

// One lane's share of one row's block: quarter kq of Q4_K (64 columns: 32
// bytes of nibbles), or of Q6_K words 4 (kq % 2) .. +3 of both ql runs and of
// qh in half kq / 2; and the header.
template <bool Q4>
struct Raw {
    uint4 q[Q4 ? 2 : 3];
    uint4 h;   // Q4_K: d, dmin, scales; Q6_K: x, y = scales of the half, z = d
};

template <int TYPE>
__device__ __forceinline__ Raw<TYPE == QK_TYPE_Q4_K> load_raw(const uint8_t *row, int b, int nb, int kq) {
    Raw<TYPE == QK_TYPE_Q4_K> r;
    if constexpr (TYPE == QK_TYPE_Q4_K) {
        const uint8_t *p = row + b * 144;
        r.h = load16(p);
        r.q[0] = load16(p + 16 + kq * 32);
        r.q[1] = load16(p + 32 + kq * 32);
    } else {
        const Q6Fields f = q6_fields(row, nb, b, TYPE == QK_TYPE_Q6_K_SPLIT);
        const int kh = kq >> 1, jh = kq & 1;
        r.q[0] = load16(f.ql + kh * 64 + 16 * jh);
        r.q[1] = load16(f.ql + kh * 64 + 32 + 16 * jh);
        r.q[2] = load16(f.qh + kh * 32 + 16 * jh);
        const uint2 sc = load8(f.sc + kh * 8);
        r.h = make_uint4(sc.x, sc.y, load2(f.d), 0);
    }
    return r;
}

// A block's activations of eight tokens: lane (n, kq) holds operand row n
// (token n % 8, high halves for n < 8, else low), the block's sub-block sums
// (Q4_K) and the scales of the four rows its accumulators belong to.
template <bool Q4>
struct Operand {
    half8 a[8];
    half4 m;
    float f[4];
};

__device__ __forceinline__ float wave_max64(float v) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

// LDS of one wave while it converts a block: the operand in reading order
// ([step][quarter][row] x 16 bytes), the sub-block sums ([quarter][row] half4)
// and the tokens' scales.
constexpr int kOperandLds = 8 * 1024, kSumLds = 512, kScratch = kOperandLds + kSumLds + 64;

// Block b of every token, four consecutive columns a lane: one 1 KB read a
// token, all in flight (a token past the last reads the last again).
__device__ __forceinline__ void load_block_input(const float *x, int ldx, int n_tokens, int b, int lane,
                                                 float4 (&v)[kSlots - 1]) {
    #pragma unroll
    for (int t = 0; t < kSlots - 1; ++t)
        v[t] = *reinterpret_cast<const float4 *>(x + static_cast<int64_t>(min(t, n_tokens - 1)) * ldx + b * 256 + 4 * lane);
}

// The block's operand from its values v, through this wave's scratch:
// stage_store_wave's arithmetic (x' = x * 2^shift with the block's maximum in
// [2^14, 2^15), fp16 high and low halves, sums of 32 values, a non-finite value
// making the token's scale NaN).  Rows of absent tokens hold anything.
template <bool Q4>
__device__ __forceinline__ void build_operand(const float4 (&v)[kSlots - 1], int n_tokens, int lane,
                                              unsigned char *scratch, Operand<Q4> &op) {
    const int kq = lane >> 4;
    // Lane l's columns 4 l .. +3: operand step, quarter and half.
    const int step = Q4 ? lane & 7 : ((lane >> 4) & 1) * 4 + (lane & 3);
    const int quarter = Q4 ? lane >> 4 : (lane >> 5) * 2 + ((lane >> 2) & 1);
    unsigned char *const at = scratch + step * 1024 + quarter * 256 + ((lane >> 3) & 1) * 8;
    unsigned char *const sums = scratch + kOperandLds;
    float *const scales = reinterpret_cast<float *>(scratch + kOperandLds + kSumLds);
    if constexpr (Q4) reinterpret_cast<uint2 *>(sums)[lane] = make_uint2(0, 0);
    #pragma unroll
    for (int t = 0; t < kSlots - 1; ++t) {
        if (t >= n_tokens) break;
        const float4 x = v[t];
        float mx = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
        int bad = !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(x.w));
        mx = wave_max64(mx);
        bad = __builtin_amdgcn_ballot_w64(bad) != 0;
        int shift = 0;
        float f = 0.f;
        if (mx > 0.f && isfinite(mx)) {
            shift = min(15 - __builtin_amdgcn_frexp_expf(mx), 140);
            f = ldexpf(1.f, -shift);
        }
        if (bad) f = __builtin_nanf("");
        const float x4[4] = {bad ? 0.f : ldexpf(x.x, shift), bad ? 0.f : ldexpf(x.y, shift),
                             bad ? 0.f : ldexpf(x.z, shift), bad ? 0.f : ldexpf(x.w, shift)};
        half4 h, l;
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = i == 1 ? 2 : i == 2 ? 1 : i;   // byte order 0, 2, 1, 3
            h[e] = static_cast<_Float16>(x4[i]);
            l[e] = static_cast<_Float16>(x4[i] - static_cast<float>(h[e]));
        }
        *reinterpret_cast<half4 *>(at + t * 16) = h;
        *reinterpret_cast<half4 *>(at + (8 + t) * 16) = l;
        if constexpr (Q4) {
            float sum = (x4[0] + x4[1]) + (x4[2] + x4[3]);
            sum += __shfl_xor(sum, 1);
            sum += __shfl_xor(sum, 2);
            sum += __shfl_xor(sum, 4);
            if ((lane & 7) == 0) {
                // Sub-block lane / 8 at K = 4 (sub / 2) + sub % 2, / 64 to stay
                // inside the fp16 range.
                const float s64 = sum * (1.f / 64.f);
                const _Float16 sh = static_cast<_Float16>(s64);
                _Float16 *m = reinterpret_cast<_Float16 *>(sums) + (lane >> 4) * 64 + ((lane >> 3) & 1);
                m[t * 4] = sh;
                m[(8 + t) * 4] = static_cast<_Float16>(s64 - static_cast<float>(sh));
            }
        }
        if (lane == 0) scales[t] = f;
    }
    // This wave's own stores: in order with its reads.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    #pragma unroll
    for (int s = 0; s < 8; ++s) op.a[s] = *reinterpret_cast<const half8 *>(scratch + s * 1024 + lane * 16);
    if constexpr (Q4) op.m = reinterpret_cast<const half4 *>(sums)[lane];
    // Accumulator r of a lane: operand row 4 kq + r, token 4 (kq % 2) + r.
    const float4 f4 = *reinterpret_cast<const float4 *>(scales + 4 * (kq & 1));
    op.f[0] = f4.x;
    op.f[1] = f4.y;
    op.f[2] = f4.z;
    op.f[3] = f4.w;
}

// acc += one block's product: the chains over both halves, scaled.
template <int TYPE>
__device__ __forceinline__ void multiply_block(const Raw<TYPE == QK_TYPE_Q4_K> &r,
                                               const Operand<TYPE == QK_TYPE_Q4_K> &op, int kq, float4v &acc) {
    constexpr bool Q4 = TYPE == QK_TYPE_Q4_K;
    float4v t = {0.f, 0.f, 0.f, 0.f};
    float d;
    if constexpr (Q4) {
        uint32_t sc4, mn4;
        q4k_scale_min4(r.h, kq >> 1, sc4, mn4);
        const int sh = 16 * (kq & 1);
        const _Float16 sa = u8_to_h(sc4 >> sh), sb = u8_to_h(sc4 >> (sh + 8));
        const half2v sa2 = h2(sa), ba2 = h2(static_cast<_Float16>(-1024.f) * sa);
        const half2v sb2 = h2(sb * static_cast<_Float16>(0.0625f)), bb2 = h2(static_cast<_Float16>(-64.f) * sb);
        #pragma unroll
        for (int s = 0; s < 8; ++s)
            t = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                op.a[s], __builtin_bit_cast(half8, decode_q4(quad_word(r.q[s >> 2], s & 3), sa2, ba2, sb2, bb2)), t, 0, 0, 0);
        d = f16_bits_to_f32(r.h.x & 0xFFFFu);
        const float dm = -64.f * f16_bits_to_f32(r.h.x >> 16);
        half4 bm;
        bm[0] = u8_to_h(mn4 >> sh);
        bm[1] = u8_to_h(mn4 >> (sh + 8));
        bm[2] = bm[3] = static_cast<_Float16>(0.f);
        float4v tm = {0.f, 0.f, 0.f, 0.f};
        tm = __builtin_amdgcn_mfma_f32_16x16x16f16(op.m, bm, tm, 0, 0, 0);
        #pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(dm * op.f[e], tm[e], acc[e]);
    } else {
        const int jh = kq & 1;
        bool lane_wide = false;
        #pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int s = static_cast<int8_t>(((e < 4 ? r.h.x : r.h.y) >> (8 * (e & 3))) & 0xFFu);
            lane_wide |= s > 62 || s < -62;
        }
        const bool wide = __builtin_amdgcn_ballot_w64(lane_wide) != 0;
        #pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t la = quad_word(r.q[0], s & 3), lb = quad_word(r.q[1], s & 3), hq = quad_word(r.q[2], s & 3);
            const uint32_t sw = s < 4 ? r.h.x : r.h.y;
            const half2v sa = h2(s8_to_h(sw >> (8 * jh))), sb = h2(s8_to_h(sw >> (8 * jh + 16)));
            uint4 a, b;
            if (s < 4)
                decode_q6<0>(la, lb, hq, sa, sb, a, b);
            else
                decode_q6<1>(la, lb, hq, sa, sb, a, b);
            t = __builtin_amdgcn_mfma_f32_16x16x32_f16(op.a[s], __builtin_bit_cast(half8, a), t, 0, 0, 0);
            if (wide) t = __builtin_amdgcn_mfma_f32_16x16x32_f16(op.a[s], __builtin_bit_cast(half8, b), t, 0, 0, 0);
        }
        d = f16_bits_to_f32(r.h.z);
    }
    #pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = fmaf(d * op.f[e], t[e], acc[e]);
}

template <int TYPE, int NTL, int BPW>
__device__ __forceinline__ void few_body(const FewParams &p, const FewMatrix &M, const FewMatrix &M1, int item0,
                                         float *red) {
    constexpr bool Q4 = TYPE == QK_TYPE_Q4_K;
    static_assert(BPW == 1 || NTL == 1, "two blocks a wave take one tile");
    const int lane = threadIdx.x & 63, n = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int tiles = (M.rows + kTileRows - 1) / kTileRows;
    const int per = p.pair ? 1 : NTL;                    // row tiles of M a step takes
    const int steps = (tiles + per - 1) / per;

    // Tile l of step i, clamped to the last (whose extra sums are not stored).
    auto row_of = [&](int i, int l) {
        const FewMatrix &m = p.pair && l ? M1 : M;
        const int tile = p.pair ? i : i * NTL + l;
        return m.w + static_cast<size_t>(min(tile * kTileRows + n, M.rows - 1)) * m.row_bytes;
    };
    // Wave w's blocks: w and, with two, w + waves (past the row's end the last
    // block is read again and left out).
    const bool second = wave + waves < p.nb;
    const int blk0 = wave, blk1 = min(wave + waves, p.nb - 1);
    Raw<Q4> cur[NTL], more;
    #pragma unroll
    for (int l = 0; l < NTL; ++l) cur[l] = load_raw<TYPE>(row_of(min(item0, steps - 1), l), blk0, p.nb, kq);
    if constexpr (BPW == 2) more = load_raw<TYPE>(row_of(min(item0, steps - 1), 0), blk1, p.nb, kq);

    // Activations, while the first tiles are in flight.
    unsigned char *const scratch = reinterpret_cast<unsigned char *>(red) + wave * kScratch;
    float4 v[BPW][kSlots - 1];
    load_block_input(p.x, p.ldx, p.n_tokens, blk0, lane, v[0]);
    if constexpr (BPW == 2) load_block_input(p.x, p.ldx, p.n_tokens, blk1, lane, v[1]);
    if (p.norm_w) {
        #pragma unroll
        for (int t = 0; t < kSlots - 1; ++t) {
            float ss = 0.f;
            #pragma unroll
            for (int k = 0; k < BPW; ++k) {
                const float4 &x = v[k][t];
                const float part = fmaf(x.w, x.w, fmaf(x.z, x.z, fmaf(x.y, x.y, x.x * x.x)));
                ss += k && !second ? 0.f : part;
            }
            ss = wave_sum(ss);
            if (lane == 0) red[wave * kSlots + t] = ss;
        }
        __syncthreads();
        float scale[kSlots - 1];
        #pragma unroll
        for (int t = 0; t < kSlots - 1; ++t) {
            float all = 0.f;
            for (int w = 0; w < waves; ++w) all += red[w * kSlots + t];
            scale[t] = 1.0f / sqrtf(all / static_cast<float>(p.nb * 256) + p.norm_eps);
        }
        __syncthreads();
        #pragma unroll
        for (int k = 0; k < BPW; ++k) {
            const float4 w = *reinterpret_cast<const float4 *>(p.norm_w + (k ? blk1 : blk0) * 256 + 4 * lane);
            #pragma unroll
            for (int t = 0; t < kSlots - 1; ++t)
                v[k][t] = make_float4(v[k][t].x * scale[t] * w.x, v[k][t].y * scale[t] * w.y, v[k][t].z * scale[t] * w.z,
                                      v[k][t].w * scale[t] * w.w);
        }
    }
    if (p.up) {
        #pragma unroll
        for (int k = 0; k < BPW; ++k) {
            float4 u[kSlots - 1];
            load_block_input(p.up, p.ldx, p.n_tokens, k ? blk1 : blk0, lane, u);
            #pragma unroll
            for (int t = 0; t < kSlots - 1; ++t)
                v[k][t] = make_float4(silu_mul_value(v[k][t].x, u[t].x), silu_mul_value(v[k][t].y, u[t].y),
                                      silu_mul_value(v[k][t].z, u[t].z), silu_mul_value(v[k][t].w, u[t].w));
        }
    }
    Operand<Q4> op, op2;
    build_operand<Q4>(v[0], p.n_tokens, lane, scratch, op);
    if constexpr (BPW == 2) build_operand<Q4>(v[1], p.n_tokens, lane, scratch, op2);
    __syncthreads();   // the scratch becomes the sums

    // Store the step's outputs from its sums: the waves' in wave order, the
    // high and low parts already together.
    auto store = [&](int i, const float *sums) {
        const int outs = p.pair ? 128 : NTL * 128;
        for (int j = threadIdx.x; j < outs; j += blockDim.x) {
            const int l = j >> 7, t = (j >> 4) & 7;
            const int row = (p.pair ? i : i * NTL + l) * kTileRows + (j & 15);
            float sum = 0.f;
            for (int w = 0; w < waves; ++w) sum += sums[(l * waves + w) * 128 + (j & 127)];
            if (p.pair) {
                float u = 0.f;
                for (int w = 0; w < waves; ++w) u += sums[(waves + w) * 128 + (j & 127)];
                sum = silu_mul_value(sum, u);
            }
            if (t < p.n_tokens && row < M.rows) {
                float *y = M.y + static_cast<int64_t>(t) * M.ldy + row;
                *y = p.accumulate ? *y + sum : sum;
            }
        }
    };
    auto publish = [&](float4v acc, float *out) {
        // High and low parts: lanes 32 apart hold the same token.
        #pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], 32);
        if (kq < 2)
            #pragma unroll
            for (int e = 0; e < 4; ++e) out[(4 * kq + e) * 16 + n] = acc[e];
    };
    // This wave's LDS stores, then the workgroup; loads stay in flight.
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    if constexpr (BPW == 2) {
        // One step a workgroup (launch_few).
        float4v acc = {0.f, 0.f, 0.f, 0.f};
        multiply_block<TYPE>(cur[0], op, kq, acc);
        if (second) multiply_block<TYPE>(more, op2, kq, acc);
        publish(acc, red + wave * 128);
        meet();
        store(item0, red);
    } else {
        for (int i = item0, turn = 0; i < steps; i += M.blocks, turn ^= 1) {
            Raw<Q4> next[NTL];
            const int ni = min(i + M.blocks, steps - 1);   // unconditional: past the end the last again
            #pragma unroll
            for (int l = 0; l < NTL; ++l) next[l] = load_raw<TYPE>(row_of(ni, l), blk0, p.nb, kq);
            float *const sums = red + turn * NTL * waves * 128;
            #pragma unroll
            for (int l = 0; l < NTL; ++l) {
                float4v acc = {0.f, 0.f, 0.f, 0.f};
                multiply_block<TYPE>(cur[l], op, kq, acc);
                publish(acc, sums + (l * waves + wave) * 128);
            }
            // (The other turn's sums are free: their readers passed the
            // previous meeting.)
            meet();
            store(i, sums);
            #pragma unroll
            for (int l = 0; l < NTL; ++l) cur[l] = next[l];
        }
    }
}

template <int TYPE, int NTL, int BPW>
__global__ __launch_bounds__(kMaxWaves * 64) void few_gemm(FewParams p) {
    extern __shared__ __align__(16) float red[];   // the waves' scratch, then two turns of [tile][wave][token][row] sums
    int m = 0;
    if (!p.pair) {
        #pragma unroll
        for (int i = 1; i < QK_MAX_FUSED; ++i)
            m += (i < p.n_mats && static_cast<int>(blockIdx.x) >= p.mat[i].block_begin) ? 1 : 0;
    }
    m = __builtin_amdgcn_readfirstlane(m);
    const FewMatrix &M = p.mat[m], &M1 = p.mat[p.pair ? 1 : m];
    const int item0 = static_cast<int>(blockIdx.x) - M.block_begin;
    if constexpr (TYPE != 0)
        few_body<TYPE, NTL, BPW>(p, M, M1, item0, red);
    else if (M.type == QK_TYPE_Q4_K)
        few_body<QK_TYPE_Q4_K, NTL, BPW>(p, M, M1, item0, red);
    else if (M.type == QK_TYPE_Q6_K)
        few_body<QK_TYPE_Q6_K, NTL, BPW>(p, M, M1, item0, red);
    else
        few_body<QK_TYPE_Q6_K_SPLIT, NTL, BPW>(p, M, M1, item0, red);
}

template <int NTL, int BPW>
void launch_form(int type, const dim3 &grid, const dim3 &block, size_t lds, hipStream_t s, const FewParams &p) {
    if (type == QK_TYPE_Q4_K)
        hipLaunchKernelGGL((few_gemm<QK_TYPE_Q4_K, NTL, BPW>), grid, block, lds, s, p);
    else if (type == QK_TYPE_Q6_K)
        hipLaunchKernelGGL((few_gemm<QK_TYPE_Q6_K, NTL, BPW>), grid, block, lds, s, p);
    else if (type == QK_TYPE_Q6_K_SPLIT)
        hipLaunchKernelGGL((few_gemm<QK_TYPE_Q6_K_SPLIT, NTL, BPW>), grid, block, lds, s, p);
    else
        hipLaunchKernelGGL((few_gemm<0, NTL, BPW>), grid, block, lds, s, p);
}

}  // namespace

// Supported: rows of at most sixteen blocks, or (no pair) of 32 where every
// workgroup has one tile to take -- two blocks a wave, converted one after the
// other.  And shorter, by estimates fitted to 1 to 140 MB of each type in rows of
// 1 to 32 blocks at 2 to 7 tokens, both forms measured for each: here a base that
// grows with the waves that meet, a conversion per token and the weights (short
// rows: more of a tile's work is the meeting); one GEMV column per token the
// launch and the bytes of every token, its re-reads coming from cache (powers of
// two of blocks divide evenly over its waves).  Of the 1524 shapes measured, the
// accepted ones take 0.55 to 1.02 of the GEMV's time but for two (1.05 and 1.08).
bool few_pays(const qk_matrix *mats, int n_mats, int cols, int n_tokens, bool pair) {
    const int nb = cols / 256;
    const bool two = nb > kMaxWaves;
    if (n_tokens < 2 || n_tokens >= kSlots || nb > 2 * kMaxWaves) return false;
    if (pair && (two || n_mats != 2 || mats[0].type != mats[1].type || mats[0].rows != mats[1].rows)) return false;
    struct Cost {
        double base, block, token, mb;   // us, us a block of the row, us a token, us a MB
    };
    constexpr Cost kOne[3] = {{3.2, 0.19, 0.83, 0.22}, {4.6, 0.5, 0.5, 0.35}, {3.9, 0.25, 0.6, 0.29}};
    constexpr Cost kTwo[3] = {{7.9, 0., 1.97, 0.035}, {13.1, 0., 1.35, 0.04}, {10.1, 0., 1.58, 0.06}};
    double fixed = 0., stream = 0., mb = 0.;
    int64_t tiles = 0;
    for (int i = 0; i < n_mats; ++i) {
        const int t = mats[i].type == QK_TYPE_Q4_K ? 0 : mats[i].type == QK_TYPE_Q6_K ? 1 : 2;
        const Cost &c = two ? kTwo[t] : kOne[t];
        const double m = 1e-6 * static_cast<double>(row_bytes(mats[i].type, nb)) * mats[i].rows;
        fixed = std::max(fixed, c.base + c.block * nb + c.token * n_tokens);
        stream += (c.mb + (two ? 0. : 0.25 / (nb * nb))) * m;
        mb += m;
        tiles += (mats[i].rows + kTileRows - 1) / kTileRows;
    }
    if (two && tiles > device_info().cus) return false;
    const double bytes = mb * n_tokens;
    const double gemv = two ? 7.1 + 0.15 * bytes : nb & (nb - 1) ? 6.5 + 0.135 * bytes : 5.2 + 0.13 * bytes;
    return 1.05 * (fixed + stream) < gemv;
}

int launch_few(const qk_matrix *mats, int n_mats, const float *x, int ldx, int cols, int n_tokens, const int *ldy,
               const GemvFusion &f, hipStream_t stream, const char *where) {
    const int nb = cols / 256;
    FewParams p{};
    p.n_mats = n_mats;
    p.x = x;
    p.ldx = ldx;
    p.n_tokens = n_tokens;
    p.nb = nb;
    p.norm_w = f.norm_w;
    p.norm_eps = f.norm_eps;
    p.up = f.up;
    p.accumulate = f.accumulate;
    p.pair = f.pair;
    const int bpw = nb > kMaxWaves ? 2 : 1, waves = (nb + bpw - 1) / bpw;
    // Sixteen waves a CU at 128 registers; each matrix its share of the
    // workgroups by bytes, at least one.
    const int slots = device_info().cus * std::max(1, std::min(4, kMaxWaves / waves));
    int64_t bytes = 0, tiles = 0;
    for (int i = 0; i < n_mats; ++i) {
        if (static_cast<int64_t>(mats[i].rows) * row_bytes(mats[i].type, nb) > (int64_t(1) << 40))
            return fail(QK_ERR_LIMIT, std::string(where) + ": matrix too large");
        bytes += static_cast<int64_t>(mats[i].rows) * row_bytes(mats[i].type, nb);
        tiles += (mats[i].rows + kTileRows - 1) / kTileRows;
    }
    // Two tiles a step where every workgroup has several.
    const int ntl = p.pair || (bpw == 1 && tiles >= 2 * static_cast<int64_t>(slots)) ? 2 : 1;
    int type = mats[0].type, blocks = 0;
    for (int i = 0; i < n_mats; ++i) {
        FewMatrix &M = p.mat[i];
        M.w = static_cast<const uint8_t *>(mats[i].w);
        M.y = mats[i].y;
        M.rows = mats[i].rows;
        M.type = mats[i].type;
        M.ldy = ldy ? ldy[i] : mats[i].rows;
        M.row_bytes = row_bytes(M.type, nb);
        const int64_t mine = (M.rows + kTileRows - 1) / kTileRows;
        const int64_t steps = p.pair ? mine : (mine + ntl - 1) / ntl;
        const int64_t share = p.pair ? slots : bpw == 2 ? steps : std::max<int64_t>(1, slots * (M.rows * M.row_bytes) / bytes);
        M.block_begin = p.pair ? 0 : blocks;
        M.blocks = static_cast<int>(std::min(steps, share));
        if (!p.pair || i == 0) blocks += M.blocks;
        if (M.type != type) type = 0;
    }
    const dim3 grid(blocks), block(64 * waves);
    const size_t lds = std::max<size_t>(2 * static_cast<size_t>(ntl) * waves * 128 * sizeof(float),
                                        static_cast<size_t>(waves) * kScratch);
    if (bpw == 2)
        launch_form<1, 2>(type, grid, block, lds, stream, p);
    else if (ntl == 2)
        launch_form<2, 1>(type, grid, block, lds, stream, p);
    else
        launch_form<1, 1>(type, grid, block, lds, stream, p);
    return launch_status(where);
}

}  // namespace qk

extern "C" int qk_rule_few_tokens(const qk_matrix *mats, int n_mats, int cols, int n_tokens, int pair) {
    return qk::few_pays(mats, n_mats, cols, n_tokens, pair != 0);
}
