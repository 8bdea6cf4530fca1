// qk_tile_attention.hip - attention of prefill chunks: 16 consecutive tokens
// of a batch that continue one sequence share its cache rows.
//
// split_attention_kernel (csrc/qk_step.hip) reads a token's rows once per
// token: a 512-token chunk over 600 earlier rows read 3.6 GB through L2, 152
// us at 24 TB/s.  Here a workgroup takes 16 tokens x one KV head with all its
// query heads and reads every cache row once for them; both products run on
// the FP32 matrix instructions (v_mfma_f32_16x16x4_f32), whose operands and
// sums are fp32 as before, so the bound is their 157 TFLOP/s (34 us for that
// chunk).  Measured: that chunk (24 heads over 8 KV heads of 128) 152 -> 80.7
// us; 512 tokens from position 0, 84 -> 45 us (32 heads over 8 of 64: 51 -> 31
// us); 1024 tokens over 3072 earlier rows, 1041 -> 469 us.
//
//   * Wave (g, s) of G x S waves (S at most 4): query head g, every S-th tile
//     of 32 cache rows.  The products are taken transposed, scores S^T = K Q^T and outputs
//     O^T = V^T P^T: a lane then holds one token's scores, the softmax needs
//     two cross-lane steps, and the probabilities are the second product's
//     operand as they stand.
//   * Key and value tiles come into LDS by direct copies, each split group
//     its own: the next key tile loads while the values are multiplied, the
//     next value tile while the next scores are.  Keys are stored with their
//     16-byte chunks rotated by row (chunk ^ row % 16), so the 16 rows of an
//     operand read fall into different banks.
//   * The S partial states of a head meet in LDS (merge as in
//     split_merge_kernel) and the outputs leave through LDS, which also
//     serves the o projection's records or codes.
//
// A tile runs here when its tokens are all valid and form at most kMaxRuns
// runs of consecutive positions of one sequence, a workgroup (blockIdx.z) each;
// the other tiles' tokens go through split_attention_kernel, which decides by
// the same test.
//
// Values that are not finite: the matrix product gives every token of the tile
// probability * value of every row, 0 * value for the rows of later tokens.
// The few rows at the run's end that some token does not see are therefore
// looked at first, and if one holds such a value, it takes part as zero and
// reaches the tokens that see it after the loop.  Elsewhere the products are
// what the per-token form's are.
#include "qk_internal.h"
#include "qk_records.h"

#include <algorithm>

namespace qk {
namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kKeys = 32;            // cache rows of a tile
// Waves of a workgroup at most: 128 registers a lane at head_dim 64, 168 at 128
// (with 16 waves it spilled 33).
constexpr int max_waves(int hd) { return hd == 64 ? 16 : 12; }

struct TileAttnArgs {
    SplitAttention a;
    int groups;    // S: waves sharing a head's rows
};

// 16 bytes a lane to LDS at dst + 16 * lane (dst wave-uniform), untracked by
// the compiler's wait insertion.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void *src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ void copies_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

constexpr int kv_bytes(int hd) { return kKeys * hd * 4; }

__device__ __forceinline__ bool finite4(const float4 &v) {
    return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
}

// Zeroes what is not finite in a tile of value rows: every wave that reads the
// tile does, before it reads.
template <int HD>
__device__ __forceinline__ void clear_not_finite(unsigned char *vbuf, int lane) {
    for (int i = 0; i < kv_bytes(HD) / 1024; ++i) {
        float4 *at = reinterpret_cast<float4 *>(vbuf + i * 1024 + lane * 16);
        const float4 v = *at;
        *at = make_float4(isfinite(v.x) ? v.x : 0.f, isfinite(v.y) ? v.y : 0.f, isfinite(v.z) ? v.z : 0.f,
                          isfinite(v.w) ? v.w : 0.f);
    }
}

template <int HD>
__global__ __launch_bounds__(max_waves(HD) * 64) void tile_attention(TileAttnArgs ta) {
    extern __shared__ __align__(16) unsigned char lds[];
    const SplitAttention &a = ta.a;
    constexpr int NJ = HD / 16, NT = HD / 64;     // 16-dimension and 64-dimension steps
    constexpr int kChunks = HD / 4;               // 16-byte chunks of a row
    const int G = a.heads / a.kv_heads, S = ta.groups;
    const int lane = threadIdx.x & 63, n = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = wave % G, sg = wave / G;
    const int kvh = blockIdx.x, t0 = blockIdx.y * kAttnTile;

    const TokenTile tile = token_tile(a.desc, t0, a.n_tokens, a.cache_rows, a.max_pos, lane);
    // This workgroup's run: tokens i0 .. i1 - 1 of the tile, rows 0 .. last of
    // their sequence, of which `seen` and the ones before are all the tokens'.
    unsigned starts = tile.starts;
    for (unsigned r = blockIdx.z; r > 0; --r) starts &= starts - 1;
    if (!tile.shared || !starts) return;
    const int i0 = __builtin_ctz(starts);
    starts &= starts - 1;
    const int i1 = starts ? __builtin_ctz(starts) : min(kAttnTile, a.n_tokens - t0);
    const int last = __builtin_amdgcn_readfirstlane(__shfl(tile.pos, i1 - 1)), seen = last - (i1 - i0 - 1);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(__shfl(static_cast<int>(tile.kv_row), i0));
    const int hi = __builtin_amdgcn_readfirstlane(__shfl(static_cast<int>(tile.kv_row >> 32), i0));
    const int64_t row = static_cast<int64_t>(hi) << 32 | lo;
    const int mine = n >= i0 && n < i1 ? tile.pos : -1;   // rows this lane's token sees: 0 .. mine
    const int t = min(t0 + n, a.n_tokens - 1);
    const int64_t rs = a.head_major ? HD : static_cast<int64_t>(a.kv_heads) * HD;
    const float scale = 1.4426950408889634f / sqrtf(static_cast<float>(HD));

    float4 q[NJ];
    const float *qrow = a.q + (static_cast<int64_t>(t) * a.heads + kvh * G + g) * HD + 4 * kq;
    #pragma unroll
    for (int j = 0; j < NJ; ++j) q[j] = *reinterpret_cast<const float4 *>(qrow + 16 * j);

    float4v o[NT][4];
    #pragma unroll
    for (int x = 0; x < NT; ++x)
        #pragma unroll
        for (int i = 0; i < 4; ++i) o[x][i] = float4v{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;   // this lane's token; l over this lane's rows only

    unsigned char *const kbuf = lds + sg * 2 * kv_bytes(HD), *const vbuf = kbuf + kv_bytes(HD);
    const int64_t base = kv_offset(a.head_major, a.layer, a.cache_rows, a.kv_heads, HD, row, kvh);
    const float *kc = a.key_cache + base, *vc = a.value_cache + base;
    const int tiles = last / kKeys + 1, iters = (tiles + S - 1) / S;
    // Tiles from `edge` on hold rows that some token does not see: such a row
    // meets that token as 0 * value, so what is not finite in them (bad: there
    // is any) is zeroed there and joins after the loop.
    const int edge = (seen + 1) / kKeys;

    // 1 KB of a tile is 256 / HD rows; the group's G waves share the
    // pieces.  Rows past the last are the last again (in bounds; masked).
    auto copy_tile = [&](const float *src, unsigned char *dst, int j, bool rotate) {
        constexpr int kRowsPer = 256 / HD, kPieces = kKeys / kRowsPer;
        for (int i = g; i < kPieces; i += G) {
            const int r = i * kRowsPer + lane / kChunks, slot = lane % kChunks;
            const int chunk = rotate ? slot ^ (r & 15) : slot;
            dma16(src + static_cast<int64_t>(min(j * kKeys + r, last)) * rs + 4 * chunk, lds_address(dst + i * 1024));
        }
    };
    copy_tile(kc, kbuf, sg, true);
    bool bad = false;
    for (int i = threadIdx.x; i < (last + 1 - edge * kKeys) * kChunks; i += blockDim.x)
        bad |= !finite4(*reinterpret_cast<const float4 *>(vc + (edge * kKeys + i / kChunks) * rs + i % kChunks * 4));
    bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    int *const flags = reinterpret_cast<int *>(lds + S * 2 * kv_bytes(HD));   // one a wave
    if (lane == 0) flags[wave] = bad;
    copies_barrier();
    copy_tile(vc, vbuf, sg, false);
    bad = __builtin_amdgcn_ballot_w64(flags[lane < G * S ? lane : 0]) != 0;
    for (int it = 0; it < iters; ++it) {
        const int j = it * S + sg;
        const bool live = j < tiles;
        float4v st[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if (live) {
            // Chains of 16 products (8 at head_dim 64), added as a tree: as
            // exact as the per-token form's lane sums (2.1e-7 of float64
            // at head_dim 128; 4.8e-7 as one chain over a head).
            #pragma unroll
            for (int h = 0; h < 2; ++h) {
                float4v part[2][4];
                #pragma unroll
                for (int e = 0; e < 4; ++e) part[0][e] = part[1][e] = float4v{0.f, 0.f, 0.f, 0.f};
                #pragma unroll
                for (int x = 0; x < NJ; ++x) {
                    const float4 k =
                        *reinterpret_cast<const float4 *>(kbuf + ((h * 16 + n) * kChunks + ((4 * x + kq) ^ n)) * 16);
                    float4v(&c)[4] = part[x & 1];
                    c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.x, q[x].x, c[0], 0, 0, 0);
                    c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.y, q[x].y, c[1], 0, 0, 0);
                    c[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.z, q[x].z, c[2], 0, 0, 0);
                    c[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.w, q[x].w, c[3], 0, 0, 0);
                }
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    st[h][r] = ((part[0][0][r] + part[0][1][r]) + (part[0][2][r] + part[0][3][r])) +
                               ((part[1][0][r] + part[1][1][r]) + (part[1][2][r] + part[1][3][r]));
            }
        }
        copies_barrier();   // the values are in; every wave is done with the keys
        if (it + 1 < iters) copy_tile(kc, kbuf, j + S, true);
        if (live) {
            // Register r of half h: row j * 32 + 16 h + 4 kq + r.
            float mx = -INFINITY;
            #pragma unroll
            for (int h = 0; h < 2; ++h)
                #pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st[h][r] = j * kKeys + 16 * h + 4 * kq + r <= mine ? st[h][r] : -INFINITY;
                    mx = fmaxf(mx, st[h][r]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float mn = fmaxf(m, mx * scale);
            const float ref = mn == -INFINITY ? 0.f : mn;
            const float f = __builtin_amdgcn_exp2f(m - ref);
            m = mn;
            #pragma unroll
            for (int h = 0; h < 2; ++h)
                #pragma unroll
                for (int r = 0; r < 4; ++r) st[h][r] = __builtin_amdgcn_exp2f(fmaf(st[h][r], scale, -ref));
            l = fmaf(l, f, ((st[0][0] + st[0][1]) + (st[0][2] + st[0][3])) +
                               ((st[1][0] + st[1][1]) + (st[1][2] + st[1][3])));
            if (bad && j >= edge) clear_not_finite<HD>(vbuf, lane);
            // The tile's outputs as two chains of sixteen rows, added to the
            // head's one after the other.  With the scale inside the exponent's
            // fma, 1.27e-7 of float64 over 512 tokens from position 0 of 32
            // heads of 64, as the per-token form's; one chain over the tile and
            // scaled scores gave 1.40e-7.
            #pragma unroll
            for (int x = 0; x < NT; ++x) {
                float4v to[2][4];
                #pragma unroll
                for (int i = 0; i < 4; ++i) to[0][i] = to[1][i] = float4v{0.f, 0.f, 0.f, 0.f};
                #pragma unroll
                for (int h = 0; h < 2; ++h)
                    #pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float4 v = *reinterpret_cast<const float4 *>(
                            vbuf + ((h * 16 + 4 * kq + r) * kChunks + 16 * x + n) * 16);
                        to[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.x, st[h][r], to[h][0], 0, 0, 0);
                        to[h][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.y, st[h][r], to[h][1], 0, 0, 0);
                        to[h][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.z, st[h][r], to[h][2], 0, 0, 0);
                        to[h][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.w, st[h][r], to[h][3], 0, 0, 0);
                    }
                #pragma unroll
                for (int i = 0; i < 4; ++i)
                    #pragma unroll
                    for (int r = 0; r < 4; ++r) o[x][i][r] = fmaf(o[x][i][r], f, to[0][i][r]) + to[1][i][r];
            }
        }
        copies_barrier();   // the next keys are in; every wave is done with the values
        if (it + 1 < iters) copy_tile(vc, vbuf, j + S, false);
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // The groups' states meet, in group order.
    constexpr int kPart = 16 * HD + 32;   // floats of one wave's state: outputs, then (max, sum) per token
    float *parts = reinterpret_cast<float *>(lds);
    if (sg > 0) {
        float *mine = parts + ((sg - 1) * G + g) * kPart;
        #pragma unroll
        for (int x = 0; x < NT; ++x)
            #pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<float4v *>(mine + ((x * 4 + i) * 64 + lane) * 4) = o[x][i];
        if (kq == 0) {
            mine[16 * HD + 2 * n] = m;
            mine[16 * HD + 2 * n + 1] = l;
        }
    }
    __syncthreads();
    if (sg == 0) {
        for (int s = 1; s < S; ++s) {
            const float *other = parts + ((s - 1) * G + g) * kPart;
            const float mo = other[16 * HD + 2 * n], lo = other[16 * HD + 2 * n + 1];
            const float mn = fmaxf(m, mo), ref = mn == -INFINITY ? 0.f : mn;
            const float f = __builtin_amdgcn_exp2f(m - ref), fo = __builtin_amdgcn_exp2f(mo - ref);
            m = mn;
            l = l * f + lo * fo;
            #pragma unroll
            for (int x = 0; x < NT; ++x)
                #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4v po = *reinterpret_cast<const float4v *>(other + ((x * 4 + i) * 64 + lane) * 4);
                    #pragma unroll
                    for (int r = 0; r < 4; ++r) o[x][i][r] = fmaf(po[r], fo, o[x][i][r] * f);
                }
        }
        // The values that were zeroed, for the tokens that see them: of the
        // few rows at the run's end, p * value as the sums would have taken it.
        for (int key = edge * kKeys; bad && key <= last; ++key) {
            float sc = 0.f;
            #pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float4 k = *reinterpret_cast<const float4 *>(kc + key * rs + 16 * j + 4 * kq);
                sc = fmaf(q[j].x, k.x, fmaf(q[j].y, k.y, fmaf(q[j].z, k.z, fmaf(q[j].w, k.w, sc))));
            }
            sc += __shfl_xor(sc, 16);
            sc += __shfl_xor(sc, 32);
            const float pr = __builtin_amdgcn_exp2f(sc * scale - m);
            #pragma unroll
            for (int x = 0; x < NT; ++x)
                #pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float4 v = *reinterpret_cast<const float4 *>(vc + key * rs + 64 * x + 16 * kq + 4 * r);
                    const float v4[4] = {v.x, v.y, v.z, v.w};
                    #pragma unroll
                    for (int i = 0; i < 4; ++i)
                        o[x][i][r] = key <= mine && !isfinite(v4[i]) ? fmaf(pr, v4[i], o[x][i][r]) : o[x][i][r];
                }
        }
    }
    __syncthreads();   // the states are read: the output tile takes their place

    // Outputs [16 tokens][G * HD]: register r of (x, i) is dimension 64 x +
    // 16 kq + 4 r + i.
    float *out = reinterpret_cast<float *>(lds);
    const int width = G * HD;
    if (sg == 0) {
        #pragma unroll
        for (int x = 0; x < NT; ++x)
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<float4 *>(out + n * width + g * HD + 64 * x + 16 * kq + 4 * r) =
                    make_float4(o[x][0][r] / l, o[x][1][r] / l, o[x][2][r] / l, o[x][3][r] / l);
    }
    __syncthreads();
    const int have = i1 - i0;
    const int64_t ld = static_cast<int64_t>(a.heads) * HD;
    for (int i = threadIdx.x; i < have * (width / 4); i += blockDim.x) {
        const int at = i / (width / 4), c = i - at * (width / 4), tok = i0 + at;
        *reinterpret_cast<float4 *>(a.out + (t0 + tok) * ld + kvh * width + 4 * c) =
            *reinterpret_cast<const float4 *>(out + tok * width + 4 * c);
    }
    // The o projection's input, 256 columns of one token a wave.
    if (a.gemm_rec || a.q8_out) {
        const int per = (width + 255) / 256, waves = blockDim.x / 64;
        for (int i = wave; i < have * per; i += waves) {
            const int at = i / per, blk = i - at * per, c = blk * 256 + 4 * lane, tok = i0 + at, b = t0 + tok;
            const bool in = c < width;
            const float4 v = in ? *reinterpret_cast<const float4 *>(out + tok * width + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            if (a.gemm_rec) {
                const float vr[4] = {v.x, v.y, v.z, v.w};
                stage_store_wave(vr, lane, b % kTokTile,
                                 a.gemm_rec + (static_cast<size_t>(b / kTokTile) * (a.heads * HD / 256) + kvh * per + blk) *
                                                  kTileBytes);
            }
            if (a.q8_out && in) {
                uint32_t codes;
                const int64_t at = b * ld + kvh * width + c;
                quantize_quad_store(v, (lane & 7) == 0, &codes, a.q8_scale + at / 32);
                *reinterpret_cast<uint32_t *>(a.q8_out + at) = codes;
            }
        }
    }
}

int tile_groups(int G, int hd) { return std::max(1, std::min(4, max_waves(hd) / G)); }

}  // namespace

bool tile_attention_supported(const SplitAttention &a) {
    const int G = a.heads / a.kv_heads;
    return (a.head_dim == 64 || a.head_dim == 128) && G <= 8 && a.desc && !a.k && !a.rec_out && aligned(a.q, 16) &&
           (!a.gemm_rec || G * a.head_dim % 256 == 0) && (!a.q8_out || aligned(a.q8_out, 4));
}

namespace {

// Estimated times of both forms.  Tiles: rounds of one workgroup (16-token tile
// or run, KV head) per CU, each walking ceil(rows / 32 / S) row tiles in 2.4 us
// per wave of a SIMD at head_dim 128 (half that at 64; one query head a KV head
// leaves a SIMD one wave, 3.8 and 2.2 us), and 12 us of launch, ramp, merge and
// the other form's launch.  Per token: 6 ns a (token, KV head) and the rows
// through L2 at 20 TB/s.  Both within a fifth of what 128 to 1024 tokens of one
// sequence over 128 to 4096 rows measured (64 over 8 heads excepted, whose
// per-token form takes twice that), so the tiles have to be a tenth shorter.
double tile_us(int64_t workgroups, int heads, int kv_heads, int head_dim, int64_t max_rows, double step_factor) {
    const int G = heads / kv_heads, S = tile_groups(G, head_dim);
    const int64_t rounds = (workgroups + device_info().cus - 1) / device_info().cus;
    const int64_t steps = ((max_rows + kKeys - 1) / kKeys + S - 1) / S;
    const double step = std::max(head_dim == 64 ? 4.4 : 3.8, 2.4 * ((G * S + 3) / 4)) * head_dim / 128.;
    return 12. + static_cast<double>(rounds * steps) * step * step_factor;
}
double per_token_us(int64_t n_tokens, int kv_heads, int head_dim, int64_t rows) {
    return 6e-3 * static_cast<double>(n_tokens * kv_heads) + static_cast<double>(rows) * kv_heads * head_dim * 8. / 20e6;
}
constexpr double kMargin = 1.1;

}  // namespace

// A call whose descriptors are on the device, row-major caches.  Tokens of
// sequences of their own hold at most cache_rows rows together, so with n *
// (max_pos + 1) far beyond that they share rows, about that many to a row; each
// tile's descriptors decide.  A decode batch stays below, unless one sequence is
// many times as long as the rest.
//   * Sixteen tokens a row keep tiles to two runs, and a launch in vain costs 4
//     us; where reading the rows per token takes 100 us and more, four tokens a
//     row are enough (a cache with room to spare shows no more).
//   * A cache of more rows than one sequence may hold several: then a step takes
//     twice the time (rows 2 KB apart share few sets of an XCD's L2: 2 x 256
//     tokens over 800 rows 77 us, over the same rows 45; 4 x 128 over 600, 63).
// Measured with this rule, 24 over 8 heads of 128: 512 tokens over 1112 rows 166
// -> 82 us at 1112 to 65536 cache rows; 4 x 128 over 600 116 -> 91; 4 x 58 over
// 450 and 300 decoding sequences stay per token (53 against 54, 120 against 123).
bool tile_attention_call(int n_tokens, int max_pos, int64_t cache_rows, int heads, int kv_heads, int head_dim) {
    const int64_t rows = static_cast<int64_t>(n_tokens) * (max_pos + 1);
    const double per_token = per_token_us(n_tokens, kv_heads, head_dim, rows / 4 * 3);
    if (rows / (per_token < 100. ? 16 : 4) < cache_rows) return false;
    const int64_t wgs = static_cast<int64_t>((n_tokens + kAttnTile - 1) / kAttnTile) * kv_heads;
    return kMargin * tile_us(wgs, heads, kv_heads, head_dim, max_pos + 1, cache_rows > max_pos + 1 ? 2. : 1.) < per_token;
}

int tile_attention_mode(const qk_batch_token *desc, SplitAttention &a) {
    if (!tile_attention_supported(a)) return 0;
    int64_t tiled_rows = 0, rows = 0, max_rows = 0, workgroups = 0;
    int tiled = 0;
    a.tile_runs = 1;
    for (int t0 = 0; t0 < a.n_tokens; t0 += kAttnTile) {
        const int t1 = std::min(t0 + kAttnTile, a.n_tokens);
        int runs = 0;
        int64_t tile_rows = 0, longest = 0;
        for (int t = t0; t < t1; ++t) {
            runs += t == t0 || desc[t].kv_row != desc[t - 1].kv_row || desc[t].pos != desc[t - 1].pos + 1;
            tile_rows += desc[t].pos + 1;
            longest = std::max<int64_t>(longest, desc[t].pos + 1);
        }
        if (runs <= kMaxRuns) {
            tiled += t1 - t0;
            tiled_rows += tile_rows;
            max_rows = std::max(max_rows, longest);
            workgroups += static_cast<int64_t>(runs) * a.kv_heads;
            if (runs > 1) a.tile_runs = kMaxRuns;
        } else {
            rows += tile_rows;
        }
    }
    if (!tiled || kMargin * tile_us(workgroups, a.heads, a.kv_heads, a.head_dim, max_rows, 1.) >=
                      per_token_us(tiled, a.kv_heads, a.head_dim, tiled_rows))
        return 0;
    if (tiled == a.n_tokens) return 2;
    a.rows_hint = rows;
    return 1;
}

int launch_tile_attention(const SplitAttention &a, hipStream_t stream) {
    TileAttnArgs ta{a, 1};
    const int G = a.heads / a.kv_heads, hd = a.head_dim;
    ta.groups = tile_groups(G, hd);
    const size_t lds = std::max({static_cast<size_t>(ta.groups) * 2 * kv_bytes(hd) + sizeof(int) * max_waves(hd),
                                 static_cast<size_t>(ta.groups - 1) * G * (16 * hd + 32) * sizeof(float),
                                 static_cast<size_t>(kAttnTile) * G * hd * sizeof(float)});
    const dim3 grid(a.kv_heads, (a.n_tokens + kAttnTile - 1) / kAttnTile, a.tile_runs == 1 ? 1 : kMaxRuns),
        block(64 * G * ta.groups);
    if (hd == 64)
        hipLaunchKernelGGL(tile_attention<64>, grid, block, lds, stream, ta);
    else
        hipLaunchKernelGGL(tile_attention<128>, grid, block, lds, stream, ta);
    return launch_status("tile attention launch");
}

}  // namespace qk

extern "C" {

int qk_rule_tile_attention(int n_tokens, int max_pos, int64_t cache_rows, int heads, int kv_heads, int head_dim) {
    return qk::tile_attention_call(n_tokens, max_pos, cache_rows, heads, kv_heads, head_dim);
}

int qk_rule_tile_attention_step(const qk_batch_token *desc, int n_tokens, int heads, int kv_heads, int head_dim) {
    qk::SplitAttention a{};
    a.desc = desc;
    a.n_tokens = n_tokens;
    a.heads = heads;
    a.kv_heads = kv_heads;
    a.head_dim = head_dim;
    return qk::tile_attention_mode(desc, a);
}

}  // extern "C"
