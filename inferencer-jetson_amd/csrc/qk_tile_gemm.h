// qk_tile_gemm.h - the matrix-core GEMM of two 32-token tiles and more: the part
// of csrc/qk_batched.hip (whose launch parameters and output store it uses)
// that takes them.
//
// A workgroup of four waves takes 128 weight rows x 64 tokens x a run of
// 256-column blocks; wave w owns rows 32w .. 32w + 31 and multiplies them with
// both token tiles.  Weights never touch LDS: a lane holds the raw bytes of
// one row and block half and decodes each step's 16-byte B operand in
// registers, where it feeds both tiles' two (Q6_K with wide scales: three)
// MFMA chains.  Activations come from the packed records through LDS, half a
// block (eight MFMA steps) at a time.  The fp32 sums have two levels (kRun):
// few splits make long sums, and 32 blocks in one running sum, mins and dots
// added to it apart, took Q4_K 3072 x 8192 on 517 tokens to 3.55e-7 of float64
// and Q6_K to 2.02e-7 where more splits had given 3.37 and 1.88e-7; it is 3.33
// and 1.87e-7 with them.
//
// What the next half needs -- its activation copies (global_load_lds) and raw
// weight bytes -- is requested while a half multiplies and awaited when it
// ends: one barrier per 32 (48) MFMAs a wave.  The kernel this replaces asked
// the compiler to track its copies, which put a full wait in front of each
// block's first LDS read, held whole blocks in LDS (one workgroup per CU) and
// owned 256 rows x 64 tokens.  Two workgroups fit a CU now; either alone
// takes 2.5 us a Q4_K block, two together 2.4 us each: the CU's MFMA and
// decode work, not latency.  Measured with pack and reduction against that
// kernel: Q4_K 16384 x 3072 on 517 tokens 194 -> 134 us, Q6_K (split) 3072 x
// 8192 on 517 tokens 167 -> 113 us, Q4_K 2048 x 2048 on 480 tokens 34.0 ->
// 26.4 us, on 64 tokens 16.9 -> 14.1 us.  Tried: 256 rows x 128 tokens (one
// wave per SIMD, 512 registers: 182 / 112 / 34 us) and x 64 tokens (141 / 111
// / 28 us), and weights decoded once per workgroup into LDS for 128 tokens
// (192 / 119 us: a barrier per 32 columns).
#pragma once

#include "qk_operands.h"
#include "qk_records.h"

#include <type_traits>

namespace qk {
namespace {

constexpr int kHalfBytes = 2 * 8 * 1024;                 // one token tile's half block: hi, lo x 8 steps x 1 KB
constexpr int kTokenBytes = 2 * kTileM + kTileF;         // a tile's sub-block sums and scales

constexpr int kRun = 8;                                  // blocks of one running sum, then added to the total

// LDS: two half-block buffers of two token tiles, then two blocks' token data.
constexpr int kTileLds = 2 * 2 * (kHalfBytes + kTokenBytes);

// 1 KB from global memory (src, wave-uniform) to LDS (dst): 16 bytes a lane at
// lane16 = 16 * lane.  Inline assembly: the compiler would wait for every
// copy in flight before each LDS read.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const uint8_t *src, uint32_t lane16, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(lane16), "s"(src)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// This wave's loads, copies and LDS accesses are done; the workgroup meets.
__device__ __forceinline__ void half_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A lane's raw weight bytes for half h of a block of its row (block half
// kh: columns of the record's K order):
//   Q4_K: qs[(2 kh + h) * 32 .. +32) -- steps 8h .. 8h + 7;
//   Q6_K: words 4h .. 4h + 3 of ql's two runs and of qh -- steps 4h .. 4h + 3
//   (low nibbles), then 8 + 4h .. 8 + 4h + 3 (high nibbles).
template <bool Q4>
struct RawHalf {
    uint4 q[Q4 ? 2 : 3];
};
template <bool Q4>
__device__ __forceinline__ constexpr int half_step(int h, int s) {
    return Q4 ? 8 * h + s : (s >> 2) * 8 + 4 * h + (s & 3);
}

template <int TYPE>
__device__ __forceinline__ RawHalf<TYPE == QK_TYPE_Q4_K> load_half(const uint8_t *row, int b, int nb, int kh, int h) {
    RawHalf<TYPE == QK_TYPE_Q4_K> r;
    if constexpr (TYPE == QK_TYPE_Q4_K) {
        const uint8_t *p = row + b * 144 + 16 + (2 * kh + h) * 32;
        r.q[0] = load16(p);
        r.q[1] = load16(p + 16);
    } else {
        const Q6Fields f = q6_fields(row, nb, b, TYPE == QK_TYPE_Q6_K_SPLIT);
        r.q[0] = load16(f.ql + kh * 64 + 16 * h);
        r.q[1] = load16(f.ql + kh * 64 + 32 + 16 * h);
        r.q[2] = load16(f.qh + kh * 32 + 16 * h);
    }
    return r;
}

// Q4_K: d, dmin, scales; Q6_K: x, y = scales[kh*8 .. +8), z = d.
template <int TYPE>
__device__ __forceinline__ uint4 load_header(const uint8_t *row, int b, int nb, int kh) {
    if constexpr (TYPE == QK_TYPE_Q4_K) {
        return load16(row + b * 144);
    } else {
        const Q6Fields f = q6_fields(row, nb, b, TYPE == QK_TYPE_Q6_K_SPLIT);
        const uint2 sc = load8(f.sc + kh * 8);
        return make_uint4(sc.x, sc.y, load2(f.d), 0);
    }
}

// Scale operands of one half: Q4_K sub-blocks 2 kh + h's low and high nibbles
// (sa, ba; sb, bb as decode_q4 takes them); Q6_K the four scales of its two
// step groups.
template <bool Q4>
struct HalfScales {
    half2v a[2], b[2];
};

template <bool Q4>
__device__ __forceinline__ HalfScales<Q4> half_scales(const uint4 &hdr, int kh, int h) {
    HalfScales<Q4> s;
    if constexpr (Q4) {
        uint32_t sc4, mn4;
        q4k_scale_min4(hdr, kh, sc4, mn4);
        const _Float16 sa = u8_to_h(sc4 >> (16 * h)), sb = u8_to_h(sc4 >> (16 * h + 8));
        s.a[0] = h2(sa);
        s.a[1] = h2(static_cast<_Float16>(-1024.f) * sa);
        s.b[0] = h2(sb * static_cast<_Float16>(0.0625f));
        s.b[1] = h2(static_cast<_Float16>(-64.f) * sb);
    } else {
        #pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const uint32_t sw = hf ? hdr.y : hdr.x;
            s.a[hf] = h2(s8_to_h(sw >> (8 * h)));
            s.b[hf] = h2(s8_to_h(sw >> (8 * h + 16)));
        }
    }
    return s;
}

// t += half h of a block: eight steps of TT tiles.  A: the half's
// activations in LDS, this lane's 16 bytes of tile 0, step 0.  copy(i)
// requests piece i of the next half's activations (4 * TT pieces a wave): a
// few per step, since a burst of them stalls the wave until the memory
// pipeline has taken it.
template <bool Q4, int TT, class Copy>
__device__ __forceinline__ void multiply_half(const RawHalf<Q4> &r, const HalfScales<Q4> &sc, bool first,
                                              bool wide, const unsigned char *A, Copy copy, float16v (&t)[TT]) {
    constexpr int kCopies = 4 * TT, kPerStep = (kCopies + 5) / 6;
    float16v zero;
    #pragma unroll
    for (int k = 0; k < 16; ++k) zero[k] = 0.f;
    half8 ah[TT], al[TT], w, wb;
    auto read = [&](int st, half8 (&h)[TT], half8 (&l)[TT]) {
        #pragma unroll
        for (int u = 0; u < TT; ++u) {
            h[u] = *reinterpret_cast<const half8 *>(A + u * kHalfBytes + st * 1024);
            l[u] = *reinterpret_cast<const half8 *>(A + u * kHalfBytes + 8192 + st * 1024);
        }
    };
    auto decode = [&](int st, half8 &wa, half8 &wr) {
        if constexpr (Q4) {
            wa = __builtin_bit_cast(half8, decode_q4(quad_word(r.q[st >> 2], st & 3), sc.a[0], sc.a[1], sc.b[0], sc.b[1]));
        } else {
            uint4 a, b;
            const uint32_t la = quad_word(r.q[0], st & 3), lb = quad_word(r.q[1], st & 3), hq = quad_word(r.q[2], st & 3);
            if (st < 4)
                decode_q6<0>(la, lb, hq, sc.a[0], sc.b[0], a, b);
            else
                decode_q6<1>(la, lb, hq, sc.a[1], sc.b[1], a, b);
            wa = __builtin_bit_cast(half8, a);
            wr = __builtin_bit_cast(half8, b);
        }
    };
    read(0, ah, al);
    decode(0, w, wb);
    #pragma unroll
    for (int s = 0; s < 8; ++s) {
        // The next step's operands are read and decoded while this one
        // multiplies; nothing moves further ahead (registers).
        half8 ahn[TT], aln[TT], wn, wbn;
        const int sn = s < 7 ? s + 1 : s;
        #pragma unroll
        for (int c = s * kPerStep; c < (s + 1) * kPerStep && c < kCopies; ++c) copy(c);
        read(sn, ahn, aln);
        if (s < 7) decode(sn, wn, wbn);
        #pragma unroll
        for (int u = 0; u < TT; ++u)
            t[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[u], w, first && s == 0 ? zero : t[u], 0, 0, 0);
        #pragma unroll
        for (int u = 0; u < TT; ++u) t[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[u], w, t[u], 0, 0, 0);
        if (!Q4 && wide) {
            #pragma unroll
            for (int u = 0; u < TT; ++u) t[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[u], wb, t[u], 0, 0, 0);
        }
        if (s < 7) {
            #pragma unroll
            for (int u = 0; u < TT; ++u) {
                ah[u] = ahn[u];
                al[u] = aln[u];
            }
            w = wn;
            wb = wbn;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// acc += the finished block's chains, scaled by d and the tokens' powers of
// two, minus the Q4_K mins' part (sub-block sums times mins on the MFMA, one
// tile ahead of the tile that adds them; the two parts, each larger than their
// sum, meet before the running sum).  The fence after each tile keeps the
// compiler from holding every tile's min products at once.
template <bool Q4, int TT>
__device__ __forceinline__ void finish_block(const uint4 &hdr, const unsigned char *tok, int kh, int col,
                                             const float16v (&t)[TT], float16v (&acc)[TT]) {
    const float d = f16_bits_to_f32(Q4 ? hdr.x & 0xFFFFu : hdr.z);
    half4 bm;
    float dm = 0.f;
    if constexpr (Q4) {
        dm = -64.f * f16_bits_to_f32(hdr.x >> 16);
        uint32_t sc4, mn4;
        q4k_scale_min4(hdr, kh, sc4, mn4);
        #pragma unroll
        for (int e = 0; e < 4; ++e) bm[e] = u8_to_h(mn4 >> (8 * e));
    }
    auto min_products = [&](int u) {
        float16v tm;
        #pragma unroll
        for (int k = 0; k < 16; ++k) tm[k] = 0.f;
        if constexpr (Q4) {
            const half4 mh = reinterpret_cast<const half4 *>(tok + u * kTokenBytes)[kh * 32 + col];
            const half4 ml = reinterpret_cast<const half4 *>(tok + u * kTokenBytes + kTileM)[kh * 32 + col];
            tm = __builtin_amdgcn_mfma_f32_32x32x8f16(mh, bm, tm, 0, 0, 0);
            tm = __builtin_amdgcn_mfma_f32_32x32x8f16(ml, bm, tm, 0, 0, 0);
        }
        return tm;
    };
    float16v tm = min_products(0);
    #pragma unroll
    for (int u = 0; u < TT; ++u) {
        const float4 *fr = reinterpret_cast<const float4 *>(tok + u * kTokenBytes + 2 * kTileM) + kh * 4;
        float f[16];
        #pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = fr[q];
            f[4 * q] = v.x;
            f[4 * q + 1] = v.y;
            f[4 * q + 2] = v.z;
            f[4 * q + 3] = v.w;
        }
        float16v tn = tm;
        if (Q4 && u + 1 < TT) tn = min_products(u + 1);
        #pragma unroll
        for (int k = 0; k < 16; ++k)
            acc[u][k] = Q4 ? acc[u][k] + fmaf(d * f[k], t[u][k], dm * f[k] * tm[k]) : fmaf(d * f[k], t[u][k], acc[u][k]);
        tm = tn;
        asm volatile("" : "+v"(acc[u])::"memory");
    }
}

// One workgroup's product over one matrix: rows row0 .. row0 + 127, token
// tiles tile0 .. tile0 + TT - 1 (all exist).
template <int TYPE, int TT>
__device__ __forceinline__ void tile_gemm_body(const BatchParams &p, const BatchMatrix &M, int row0, int tile0,
                                               int split, unsigned char *lds) {
    constexpr bool Q4 = TYPE == QK_TYPE_Q4_K;
    const int lane = threadIdx.x & 63, kh = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char *const tokens = lds + 2 * TT * kHalfBytes;
    const int wrow0 = row0 + wave * 32;                  // the wave's first row
    // Rows past the matrix read its last row (and store nothing).
    const uint8_t *row = M.w + static_cast<size_t>(min(wrow0 + col, M.rows - 1)) * M.row_bytes;
    const int b0 = split * p.blocks_per_split, b1 = min(p.nb, b0 + p.blocks_per_split);

    // Piece i of a half, 1 KB: wave w copies local steps 2w, 2w + 1 of every
    // tile's two parts.
    auto copy_piece = [&](int b, int h, int i) {
        const int u = i >> 2, part = (i >> 1) & 1, s = 2 * wave + (i & 1);
        const uint8_t *rec = p.records + (static_cast<size_t>(tile0 + u) * p.nb + b) * kTileBytes;
        dma16(rec + part * kTileA + half_step<Q4>(h, s) * 1024, lane * 16,
              lds_address(lds + (h * TT + u) * kHalfBytes + part * 8192 + s * 1024));
    };
    auto copy_tokens = [&](int b, int par) {
        if (wave < TT) {
            const uint8_t *src = p.records + (static_cast<size_t>(tile0 + wave) * p.nb + b) * kTileBytes + 2 * kTileA;
            unsigned char *dst = tokens + (par * TT + wave) * kTokenBytes;
            dma16(src, lane * 16, lds_address(dst));
            if (lane < (kTokenBytes - 1024) / 16) dma16(src + 1024, lane * 16, lds_address(dst + 1024));
        }
    };

    float16v acc[TT], t[TT], total[TT];
    #pragma unroll
    for (int u = 0; u < TT; ++u)
        #pragma unroll
        for (int k = 0; k < 16; ++k) acc[u][k] = t[u][k] = total[u][k] = 0.f;

    #pragma unroll
    for (int i = 0; i < 4 * TT; ++i) copy_piece(b0, 0, i);
    copy_tokens(b0, 0);
    uint4 hdr = load_header<TYPE>(row, b0, p.nb, kh);
    RawHalf<Q4> cur = load_half<TYPE>(row, b0, p.nb, kh, 0);
    half_barrier();
    for (int b = b0; b < b1; ++b) {
        const int par = (b - b0) & 1, bn = min(b + 1, b1 - 1);   // the last block requests itself again (in bounds)
        // Q6_K with a scale beyond +-62 in any of the wave's rows: the third
        // chain (wave-uniform).
        bool wide = false;
        if constexpr (!Q4) {
            bool lane_wide = false;
            #pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int s = static_cast<int8_t>(((k < 4 ? hdr.x : hdr.y) >> (8 * (k & 3))) & 0xFFu);
                lane_wide |= s > 62 || s < -62;
            }
            wide = __builtin_amdgcn_ballot_w64(lane_wide) != 0;
        }
        uint4 hdr_next = hdr;
        #pragma unroll
        for (int h = 0; h < 2; ++h) {
            RawHalf<Q4> next;
            if (h == 0) {
                next = load_half<TYPE>(row, b, p.nb, kh, 1);
            } else {
                copy_tokens(bn, par ^ 1);
                hdr_next = load_header<TYPE>(row, bn, p.nb, kh);
                next = load_half<TYPE>(row, bn, p.nb, kh, 0);
            }
            multiply_half<Q4, TT>(cur, half_scales<Q4>(hdr, kh, h), h == 0, wide, lds + h * TT * kHalfBytes + lane * 16,
                                  [&](int i) { copy_piece(h == 0 ? b : bn, h ^ 1, i); }, t);
            if (h == 1) finish_block<Q4, TT>(hdr, tokens + par * TT * kTokenBytes, kh, col, t, acc);
            half_barrier();
            cur = next;
        }
        hdr = hdr_next;
        if ((b - b0) % kRun == kRun - 1 || b + 1 == b1) {
            #pragma unroll
            for (int u = 0; u < TT; ++u) {
                total[u] += acc[u];
                #pragma unroll
                for (int k = 0; k < 16; ++k) acc[u][k] = 0.f;
            }
        }
    }

    // Accumulator register k holds token 8*(k/4) + 4*kh + k%4 of its tile.
    const int r = wrow0 + col;
    #pragma unroll
    for (int u = 0; u < TT; ++u) {
        const int tile = tile0 + u;
        if (!p.partials) {
            if (r >= M.rows) continue;
            #pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int tok = tile * kTokTile + 8 * (k >> 2) + 4 * kh + (k & 3);
                if (tok < p.n_tokens) store_out(p, M.y + static_cast<int64_t>(tok) * M.ldy + r, total[u][k]);
            }
        } else {
            const size_t slot = static_cast<size_t>(M.group_begin + row0 / kGroupRows) * p.tiles + tile;
            float *mine = p.partials + (slot * p.splits + split) * kPartialFloats + wave * 1024 + lane;
            #pragma unroll
            for (int k = 0; k < 16; ++k) mine[k * 64] = total[u][k];
        }
    }
}

// In xcd_item's list the token groups of one row group are neighbours: they share
// its weight bytes.
template <int TYPE>
__global__ __launch_bounds__(256, 2) void tile_gemm(BatchParams p, int groups, int tgroups) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int item = xcd_item(static_cast<int>(blockIdx.x), groups * tgroups * p.splits);
    if (item < 0) return;
    const int tgroup = item % tgroups, rest = item / tgroups;
    const int split = rest % p.splits, group = rest / p.splits;
    int m = 0;
    #pragma unroll
    for (int i = 1; i < QK_MAX_FUSED; ++i) m += (i < p.n_mats && group >= p.mat[i].group_begin) ? 1 : 0;
    m = __builtin_amdgcn_readfirstlane(m);
    const BatchMatrix &M = p.mat[m];
    const int row0 = (group - M.group_begin) * kGroupRows, tile0 = tgroup * 2;
    const int type = TYPE ? TYPE : M.type;
    // A ragged last group of one tile does the work of one.
    const bool both = tile0 + 1 < p.tiles;
    auto run = [&](auto t) {
        if (both)
            tile_gemm_body<decltype(t)::value, 2>(p, M, row0, tile0, split, lds);
        else
            tile_gemm_body<decltype(t)::value, 1>(p, M, row0, tile0, split, lds);
    };
    if constexpr (TYPE != 0) {
        run(std::integral_constant<int, TYPE>{});
    } else if (type == QK_TYPE_Q4_K) {
        run(std::integral_constant<int, QK_TYPE_Q4_K>{});
    } else if (type == QK_TYPE_Q6_K) {
        run(std::integral_constant<int, QK_TYPE_Q6_K>{});
    } else {
        run(std::integral_constant<int, QK_TYPE_Q6_K_SPLIT>{});
    }
}

}  // namespace
}  // namespace qk
