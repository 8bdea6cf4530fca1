// qk_operands.h - raw Q4_K / Q6_K words as exact fp16 MFMA operands, shared by
// the matrix-core GEMMs.
//
// A weight's integer part -- sc * q (Q4_K, 0..945) or s * (code - 32) (Q6_K)
// -- is exact in fp16 up to 2048 in magnitude; a Q6_K weight beyond that (a
// scale outside +-62) is the pair W_a + W_b, its rounded value and the exact
// residual.  The eight weights of an operand come from one word (Q4_K) or one
// word of each ql run (Q6_K): four from low nibbles / the first run in the
// order of bytes 0, 2, 1, 3, then four from high nibbles / the second run.
#pragma once

#include "qk_internal.h"

namespace qk {

// The hardware deals consecutive workgroups to the eight XCDs in turn: workgroup w
// of a grid of ceil(total / 8) * 8 takes item (w % 8) * ceil(total / 8) + w / 8 of a
// list, so that neighbours in the list run on one XCD and share what they read
// through its L2.  -1: none.
__device__ __forceinline__ int xcd_item(int workgroup, int total) {
    const int per = (total + 7) / 8, place = workgroup >> 3, item = (workgroup & 7) * per + place;
    return item < total && place < per ? item : -1;
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ _Float16 u8_to_h(uint32_t v) { return static_cast<_Float16>(static_cast<float>(v & 0xFFu)); }
__device__ __forceinline__ _Float16 s8_to_h(uint32_t v) {
    return static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(v & 0xFFu)));
}

__device__ __forceinline__ uint32_t quad_word(const uint4 &q, int i) {
    return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w;
}

__device__ __forceinline__ half2v h2(_Float16 v) { return half2v{v, v}; }

// (v >> S) & mask as two 16-bit lanes OR'd onto 0x6400: the fp16 values 1024 +
// bits (S negative shifts left).
template <int S>
__device__ __forceinline__ uint32_t shift_by(uint32_t v) {
    if constexpr (S >= 0) return v >> S;
    else return v << -S;
}
__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

// Eight Q4_K weights sc * q of one word: bytes (0, 2), (1, 3) low nibbles with
// scale sa, then the high nibbles with sb, each fma(1024 + n, sa, -1024 sa) or
// fma(1024 + 16 n, sb / 16, -64 sb), exact.
__device__ __forceinline__ uint4 decode_q4(uint32_t w, half2v sa, half2v ba, half2v sb, half2v bb) {
    const uint32_t w8 = w >> 8;
    uint4 o;
    o.x = as_u32(__builtin_elementwise_fma(as_h2((w & 0x000F000Fu) | 0x64006400u), sa, ba));
    o.y = as_u32(__builtin_elementwise_fma(as_h2((w8 & 0x000F000Fu) | 0x64006400u), sa, ba));
    o.z = as_u32(__builtin_elementwise_fma(as_h2((w & 0x00F000F0u) | 0x64006400u), sb, bb));
    o.w = as_u32(__builtin_elementwise_fma(as_h2((w8 & 0x00F000F0u) | 0x64006400u), sb, bb));
    return o;
}

// One pair of Q6_K weights: 6-bit code = low 4 bits of lo >> SL, 2 bits of
// hq >> SH; a = fp16(s * (code - 32)), b the exact residual.
template <int SL, int SH>
__device__ __forceinline__ void decode_q6_pair(uint32_t lo, uint32_t hq, half2v s, uint32_t &a, uint32_t &b) {
    const uint32_t n = (shift_by<SL>(lo) & 0x000F000Fu) | 0x64006400u;
    const uint32_t v = (shift_by<SH - 4>(hq) & 0x00300030u) | n;
    const half2v c = as_h2(v) + h2(static_cast<_Float16>(-1056.f));   // 1024 + code - 1056
    const half2v w = c * s;
    a = as_u32(w);
    b = as_u32(__builtin_elementwise_fma(c, s, -w));
}

template <int HF>
__device__ __forceinline__ void decode_q6(uint32_t la, uint32_t lb, uint32_t hq, half2v sa, half2v sb, uint4 &a,
                                          uint4 &b) {
    decode_q6_pair<4 * HF, 4 * HF>(la, hq, sa, a.x, b.x);
    decode_q6_pair<4 * HF + 8, 4 * HF + 8>(la, hq, sa, a.y, b.y);
    decode_q6_pair<4 * HF, 4 * HF + 2>(lb, hq, sb, a.z, b.z);
    decode_q6_pair<4 * HF + 8, 4 * HF + 10>(lb, hq, sb, a.w, b.w);
}

}  // namespace qk
