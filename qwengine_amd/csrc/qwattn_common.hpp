// Device-side helpers shared by the gated-attention kernels (gfx950 only).
//
// Model shape constants, fp16 packing, the quantized-row unpackers that turn Q8_0 / Q4_0 / F16 KV bytes into fp16
// MFMA operands, and wave64 reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qwattn.h"
#include "shapes.hpp"

namespace qwa {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int value_bytes(int kvt) {
    return kvt == QWA_KV_F16 ? 512 : kvt == QWA_KV_Q8_0 ? 256 : kvt == QWA_KV_Q4_0 ? 128 : 0;
}

__device__ __forceinline__ uint32_t h2_bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2 bits_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint16_t f2h_bits(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
__device__ __forceinline__ float h2f_bits(uint16_t u) { return (float)__builtin_bit_cast(_Float16, u); }
__device__ __forceinline__ h2 scale_pair(uint16_t a, uint16_t b) { return bits_h2((uint32_t)a | ((uint32_t)b << 16)); }

__device__ __forceinline__ h4 make_h4(uint32_t w0, uint32_t w1) {
    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
    u2v u = {w0, w1};
    return __builtin_bit_cast(h4, u);
}
__device__ __forceinline__ h8 make_h8(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    u4v u = {w0, w1, w2, w3};
    return __builtin_bit_cast(h8, u);
}

// ---- fp16 from small integers by the exponent trick: the half 0x6400 | x is 1024 + x for x < 1024, so one packed
// subtraction recovers x exactly; one packed multiply by the fp16 block scale then rounds once (the same value as
// fp16(d * x) computed in fp32).

// Q4_0 word (8 codes, element 2i in the low nibble of byte i) -> 4 half2 {(c - 8) * d} in the order
// [e0,e4], [e1,e5], [e2,e6], [e3,e7].
__device__ __forceinline__ void q4_word_to_h8(uint32_t w, h2 d, uint32_t* out) {
    const h2 bias = {(_Float16)1032.0f, (_Float16)1032.0f};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t x = ((w >> (4 * k)) & 0x000F000Fu) | 0x64006400u;
        out[k] = h2_bits((bits_h2(x) - bias) * d);
    }
}

// Q8_0: 4 int8 (one word) -> 2 half2 {x0, x1} * d, {x2, x3} * d.
__device__ __forceinline__ void q8_word_to_h4(uint32_t w, h2 d, uint32_t* out) {
    const h2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};  // 1024 + 128
    const uint32_t u = w ^ 0x80808080u;                       // biased bytes x + 128
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x05010400u);  // bytes {u0, 0x64, u1, 0x64}
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x05030402u);  // bytes {u2, 0x64, u3, 0x64}
    out[0] = h2_bits((bits_h2(lo) - bias) * d);
    out[1] = h2_bits((bits_h2(hi) - bias) * d);
}

// ---- wave64 reductions (every lane active)
// lane moves inside a row of 16 lanes (DPP, no LDS round trip): quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror (lane i
// <-> 7 - i) and row_mirror (i <-> 15 - i), which meet the lanes at distance 4 and 8 once quads and octets agree
template <int CTRL>
__device__ __forceinline__ float row_move(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
// reductions over the 32-lane half of a wave that holds one quant block, and over the wave.  (A sum over the wave through
// LDS permutes is six dependent round trips: with them the GEMV at 6144 -> 5120 took 7.05 us instead of 6.9 for one
// column, IQ3_S 15.8 instead of 12.4 for four.)
__device__ __forceinline__ float half_max(float v) {
    v = fmaxf(v, row_move<0xB1>(v));
    v = fmaxf(v, row_move<0x4E>(v));
    v = fmaxf(v, row_move<0x141>(v));
    v = fmaxf(v, row_move<0x140>(v));
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float half_sum(float v) {
    v += row_move<0xB1>(v);
    v += row_move<0x4E>(v);
    v += row_move<0x141>(v);
    v += row_move<0x140>(v);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float wave_max(float v) {
    v = half_max(v);
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
// sums: lane distances 32, 16, 8, 4, 2, 1, a fixed tree, as codes are quantized from what it feeds.  (A rotation of a row
// by 8 or 4, 0x128 and 0x124, meets the lane at that distance: all of a row for 8, and for 4 once the lanes 8 apart agree.)
__device__ __forceinline__ float half_tree(float v) {
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    v += row_move<0x128>(v);
    v += row_move<0x124>(v);
    v += row_move<0x4E>(v);
    return v + row_move<0xB1>(v);
}
__device__ __forceinline__ float wave_sum(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return half_tree(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}
// sum of y * y in lanes 0 .. 31, the first step as one FMA: y^2 of lane i + 32 rounded, that of lane i not
__device__ __forceinline__ float wave_sum_sq_low(float y) {
    const uint32_t p = __float_as_uint(y * y);
    const auto a = __builtin_amdgcn_permlane32_swap(p, p, false, false);
    return half_tree(fmaf(y, y, __uint_as_float(a[1])));
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + __expf(-x)); }

}  // namespace qwa
