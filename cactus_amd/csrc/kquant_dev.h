// Integer helpers of the K-quant GEMMs: packed 16-bit products and their split into two signed int8 digits.
#pragma once
#include "dev_common.h"

namespace chip {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// two independent 16-bit multiply-adds per dword (v_pk_mad_u16)
__device__ __forceinline__ uint32_t pk_mad16(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}
__device__ __forceinline__ uint32_t splat16(uint32_t v) { return (v & 0xffffu) | (v << 16); }

// (a & m) | (b & ~m) as one full-rate instruction
__device__ __forceinline__ uint32_t merge_bits(uint32_t m, uint32_t a, uint32_t b) { return __builtin_amdgcn_bitop3_b32(a, b, m, 0xe4); }
// four 6- to 8-bit values (bytes of v, masked by m) times a signed scale: p = v * sc + bias - 128 = 256 * hi + lo with both
// digits signed bytes.  mul = the scale, add = 128 plus the product's own bias, both in two 16-bit halves.
__device__ __forceinline__ void byte_digits(uint32_t v, uint32_t m, uint32_t mul, uint32_t add, uint32_t &hi, uint32_t &lo) {
    const uint32_t ue = pk_mad16(v & m, mul, add), uo = pk_mad16((v >> 8) & m, mul, add);
    hi = __builtin_amdgcn_perm(uo, ue, 0x07030501u);
    lo = __builtin_amdgcn_perm(uo, ue, 0x06020400u) ^ 0x80808080u;
}

// four code indices (one per byte) -> code point + 128 of kvalues_iq4nl (reference ggml-common.h), 1..241
__device__ __forceinline__ uint32_t iq4_codes(uint32_t idx) {
    constexpr uint32_t F = 0x80808080u, T0 = 0xbfad9881u ^ F, T1 = 0xf6eaddcfu ^ F, T2 = 0x26190d01u ^ F, T3 = 0x71594535u ^ F;
    const uint32_t sel = idx & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
    const uint32_t m = ((idx >> 3) & 0x01010101u) * 0xffu;
    return (lo & ~m) | (hi & m);
}
// scale of sub-block ib of IQ4_XS, -32..31, from d | scales_h | scales_l
__device__ __forceinline__ int iq4_xs_scale(const u32x2 &h, int ib) {
    return (int)(((h.y >> (4 * ib)) & 15u) | (((h.x >> (16 + 2 * ib)) & 3u) << 4)) - 32;
}

}  // namespace chip
