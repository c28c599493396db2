// Integer helpers of the K-quant GEMMs: packed 16-bit products and their split into two signed int8 digits.
#pragma once
#include "dev_common.h"

namespace chip {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// two independent 16-bit products / multiply-adds per dword (v_pk_mul_lo_u16, v_pk_mad_u16)
__device__ __forceinline__ uint32_t pk_mul16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
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

}  // namespace chip
