// Prefill GEMM for gfx950 over K-quant weights (Q2_K .. Q6_K, IQ4_XS) and Q8_K activations: the batched form of
// lm_ggml_vec_dot_q2_K_q8_K .. _q6_K_q8_K, _iq4_xs_q8_K (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// Per 256-value super-block the reference forms two integers per (row, token),
//     sumi = sum_j sc_j * dot(q_j, a_j)        and (Q4_K, Q5_K)        summ = sum_j m_j * bsum_j,
// with 6-bit (Q4_K, Q5_K: 32-value sub-blocks) or 8-bit signed (Q6_K: 16-value sub-blocks) integer sub-block
// scales, and applies the fp16 super-block scales d, dmin and the fp32 activation scale once per super-block.
// Applying an integer scale after each 32-value MFMA would cost vector work per integer sum, which is what bounds
// the Q4_0 GEMM.  Here the integer scales are folded into the int8 MFMA operand instead, as two digit planes:
//
//   Q4_K   sc = 8*sh + sl (3-bit digits): planes q*sh and q*sl (both <= 105), sumi = 8*P0 + P1
//   Q5_K   the same digits on (q - 16) in -16..15 (products in -112..105), sumi = 8*P0 + P1 + 16 * sum_j sc_j * bsum_j
//   Q3_K   (4 - q)*sc (q = 0..7, sc = -32..31) lies in -128..124: one plane, sumi = -P0
//   Q2_K   q*sc <= 45: one plane, sumi = P0; its sixteen mins stand against one bsum each in the fp16 product below
//   IQ4_XS (code point)*sc + 4064 in 127..8128: the two digits of Q6_K's form
//   Q6_K   (q - 32)*sc + 4064 = 64*hi + lo with hi in 0..127, lo in 0..63: the digits of the biased product,
//          sumi = 64*P0 + P1 - 4064 * (sum of the token's 256 quants, i.e. of its 16 bsums)
//
// so both planes accumulate in the MFMA's own int32 accumulator over the 8 k-blocks of a super-block.  The sums
// against the activation block sums, summ (and Q5_K's sum_j sc_j * bsum_j), are a product with inner dimension 16
// per super-block - the 16 bsums of block_q8_K, each |bsum| <= 2048, against m_j (sc_j) <= 63 taken twice - which
// is exact in fp16 inputs with fp32 accumulation: one v_mfma_f32_32x32x16_f16 per super-block and tile.  The vector
// unit works only once per super-block and output (5-6 operations per 256 values instead of 16).  All sums are
// exact integers, equal to the reference's sumi and summ.
//
// Structure: a workgroup of WR x WC waves owns 32*WR rows x 64*WC tokens; each wave owns one 32-row tile by two
// 32-token tiles.  LDS is double buffered over stages of 4 k-blocks (half a super-block), one barrier per stage.
// Operand cells are 16 bytes ([plane][k-block][k-half][row]), exactly what one lane feeds v_mfma_i32_32x32x32_i8.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace chip {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int KQ_KB = 4;                      // 32-value k-blocks per LDS stage
constexpr int KQ_TN = 2;                      // 32-token tiles per wave
constexpr int Q6_BIAS = 4064;                 // 32 * 127: makes (q - 32) * sc + bias >= 0 for every int8 sc; IQ4_XS: -127..113 times -32..31

// two independent 16-bit products / multiply-adds per dword (v_pk_mul_lo_u16, v_pk_mad_u16)
__device__ __forceinline__ uint32_t pk_mul16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_mad16(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}
__device__ __forceinline__ uint32_t splat16(uint32_t v) { return (v & 0xffffu) | (v << 16); }

// 6-bit scales and mins of sub-blocks 2jp and 2jp+1 (low byte, next byte) from the 12 packed bytes that follow
// d and dmin (reference ggml-quants.c:625-632); uniform branch: jp < 2 for the first half of a super-block
__device__ __forceinline__ void scale_min_pair(const u32x4 &h, int jp, uint32_t &sc, uint32_t &mn) {
    const int sh = 16 * (jp & 1);
    const uint32_t a1 = h.y >> sh, a2 = h.z >> sh, a3 = h.w >> sh;
    if (jp < 2) { sc = a1 & 0x3f3fu; mn = a2 & 0x3f3fu; }
    else        { sc = (a3 & 0x0f0f0f0fu & 0xffffu) | ((a1 >> 2) & 0x3030u); mn = ((a3 >> 4) & 0x0f0fu) | ((a2 >> 2) & 0x3030u); }
}
// the same for four sub-blocks at once, one per byte: sub-blocks 0..3 (g = 0) or 4..7 (g = 1)
__device__ __forceinline__ void scale_min_quad(const u32x4 &h, int g, uint32_t &sc, uint32_t &mn) {
    if (g == 0) { sc = h.y & 0x3f3f3f3fu; mn = h.z & 0x3f3f3f3fu; }
    else        { sc = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u); mn = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u); }
}
// four small integers (one per byte) -> the fp16 operand cell {b0, b0, b1, b1, b2, b2, b3, b3}: sub-block j stands
// against the two 16-value bsums 2j and 2j+1
__device__ __forceinline__ u32x4 bytes_to_f16_pairs(uint32_t v) {
    u32x4 c;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t hbits = (uint32_t)__half_as_ushort(__float2half_rn((float)((v >> (8 * i)) & 0xffu)));   // exact
        c[i] = hbits | (hbits << 16);
    }
    return c;
}
// eight int16 -> eight fp16 (exact for |v| <= 2048)
__device__ __forceinline__ u32x4 i16x8_to_f16(const u32x4 &v) {
    u32x4 c;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const _Float16 lo = (_Float16)(int16_t)(v[i] & 0xffffu), hi = (_Float16)(int16_t)(v[i] >> 16);
        c[i] = (uint32_t)__builtin_bit_cast(unsigned short, lo) | ((uint32_t)__builtin_bit_cast(unsigned short, hi) << 16);
    }
    return c;
}

// One staging item = (row, x) of a stage h (half of a super-block): 16 bytes of packed quants that expand into
// the 16-value k-half hf = x & 1 of two k-blocks kb0(x), kb1(x) of the stage, for both digit planes.
struct Emit {
    u32x4 cell[2][2];      // [plane][0: k-block kb0, 1: k-block kb1]  (IQ4_XS: the two k-halves of k-block x)
};
// LDS position [k-block][k-half] of an item's two cells
template <class T> __device__ __forceinline__ int cell_pos(int x, int c) {
    if constexpr (T::HALVES) return 2 * x + c;
    else return (c ? T::kb1(x) : T::kb0(x)) * 2 + (x & 1);
}

template <int WT> struct KQ;

template <> struct KQ<T_Q4_K> {
    static constexpr int BYTES = BYTES_Q4_K, NF16 = 1;             // fp16 products: summ
    static constexpr int NPL = 2;                                  // int8 digit planes
    static constexpr bool HALVES = false;
    static constexpr bool HAS_BSUM = false;
    // what item x of a row needs from one super-block: the 16 header bytes and 16 quant bytes per half
    struct Raw { u32x4 hdr, q[2]; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        r.hdr = *reinterpret_cast<const u32x4 *>(blk);
        r.q[0] = *reinterpret_cast<const u32x4 *>(blk + 16 + 16 * x);             // qs[32*jp + 16*hf], jp = 2h + x/2
        r.q[1] = *reinterpret_cast<const u32x4 *>(blk + 80 + 16 * x);
    }
    __device__ static __forceinline__ int kb0(int x) { return x & 2; }            // low nibbles: sub-block 2*jp
    __device__ static __forceinline__ int kb1(int x) { return (x & 2) + 1; }      // high nibbles: sub-block 2*jp + 1
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        uint32_t sc, mn;
        scale_min_pair(r.hdr, 2 * h + (x >> 1), sc, mn);
        const uint32_t sc0 = sc & 0xff, sc1 = sc >> 8;
        const uint32_t sh0 = splat16(sc0 >> 3), sl0 = splat16(sc0 & 7), sh1 = splat16(sc1 >> 3), sl1 = splat16(sc1 & 7);
        const u32x4 q = r.q[h];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = q[i] & 0x0f0f0f0fu, hi = (q[i] >> 4) & 0x0f0f0f0fu;
            e.cell[0][0][i] = pk_mul16(lo, sh0); e.cell[1][0][i] = pk_mul16(lo, sl0);   // byte products < 256: no carries
            e.cell[0][1][i] = pk_mul16(hi, sh1); e.cell[1][1][i] = pk_mul16(hi, sl1);
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.hdr.x; }        // d | dmin << 16
    // fp16 operand cell of item x < 2: mins of sub-blocks 4x .. 4x+3
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &r, int x) {
        uint32_t sc, mn;
        scale_min_quad(r.hdr, x & 1, sc, mn);
        return bytes_to_f16_pairs(mn);
    }
    __device__ static __forceinline__ float value(int p0, int p1, const float (&f)[2], uint32_t dd, int) {
        return __builtin_fmaf(-h2f(dd >> 16), f[0], __builtin_fmaf(h2f(dd), (float)((p0 << 3) + p1), 0.f));
    }
};

template <> struct KQ<T_Q5_K> {
    static constexpr int BYTES = BYTES_Q5_K, NF16 = 2;             // fp16 products: summ, sum_j sc_j * bsum_j
    static constexpr int NPL = 2;                                  // int8 digit planes
    static constexpr bool HALVES = false;
    static constexpr bool HAS_BSUM = false;
    struct Raw { u32x4 hdr, qh, q[2]; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        r.hdr = *reinterpret_cast<const u32x4 *>(blk);
        r.qh = *reinterpret_cast<const u32x4 *>(blk + 16 + 16 * (x & 1));          // qh[l], l = 16*hf + [0,16)
        r.q[0] = *reinterpret_cast<const u32x4 *>(blk + 48 + 16 * x);
        r.q[1] = *reinterpret_cast<const u32x4 *>(blk + 112 + 16 * x);
    }
    __device__ static __forceinline__ int kb0(int x) { return x & 2; }
    __device__ static __forceinline__ int kb1(int x) { return (x & 2) + 1; }
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        const int jp = 2 * h + (x >> 1);
        uint32_t sc, mn;
        scale_min_pair(r.hdr, jp, sc, mn);
        const uint32_t sc0 = sc & 0xff, sc1 = sc >> 8;
        // byte = q*s + (128 - 16*s) lies in 16..233 for q in 0..31, s in 0..7: no carries between the bytes of a
        // 16-bit lane, and flipping bit 7 turns it into the signed byte (q - 16)*s
        const uint32_t sh0 = sc0 >> 3, sl0 = sc0 & 7, sh1 = sc1 >> 3, sl1 = sc1 & 7;
        const uint32_t mh0 = splat16(sh0), ml0 = splat16(sl0), mh1 = splat16(sh1), ml1 = splat16(sl1);
        const uint32_t ah0 = splat16((128 - 16 * sh0) * 0x101u), al0 = splat16((128 - 16 * sl0) * 0x101u);
        const uint32_t ah1 = splat16((128 - 16 * sh1) * 0x101u), al1 = splat16((128 - 16 * sl1) * 0x101u);
        const u32x4 q = r.q[h];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // bit 2*jp of qh[l] is the fifth bit of element 64*jp + l, bit 2*jp + 1 that of 64*jp + 32 + l
            // (reference ggml-quants.c:1460-1478)
            const uint32_t hb = r.qh[i] >> (2 * jp);
            const uint32_t lo = (q[i] & 0x0f0f0f0fu) | ((hb << 4) & 0x10101010u);
            const uint32_t hi = ((q[i] >> 4) & 0x0f0f0f0fu) | ((hb << 3) & 0x10101010u);
            e.cell[0][0][i] = pk_mad16(lo, mh0, ah0) ^ 0x80808080u; e.cell[1][0][i] = pk_mad16(lo, ml0, al0) ^ 0x80808080u;
            e.cell[0][1][i] = pk_mad16(hi, mh1, ah1) ^ 0x80808080u; e.cell[1][1][i] = pk_mad16(hi, ml1, al1) ^ 0x80808080u;
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.hdr.x; }
    // item x: x / 2 = 0 mins, 1 scales; x & 1 = sub-blocks 0..3 or 4..7
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &r, int x) {
        uint32_t sc, mn;
        scale_min_quad(r.hdr, x & 1, sc, mn);
        return bytes_to_f16_pairs((x & 2) ? sc : mn);
    }
    __device__ static __forceinline__ float value(int p0, int p1, const float (&f)[2], uint32_t dd, int) {
        const int sumi = (p0 << 3) + p1 + ((int)f[1] << 4);                 // f[1] is an exact integer below 2^24
        return __builtin_fmaf(-h2f(dd >> 16), f[0], __builtin_fmaf(h2f(dd), (float)sumi, 0.f));
    }
};

template <> struct KQ<T_Q6_K> {
    static constexpr int BYTES = BYTES_Q6_K, NF16 = 0;
    static constexpr int NPL = 2;                                  // int8 digit planes
    static constexpr bool HALVES = false;
    static constexpr bool HAS_BSUM = true;
    struct Raw { u32x4 ql[2], qh[2], sc; uint32_t d; };
    // Half h of a super-block holds, for l = 0..31, the elements 128h + 32b + l of k-blocks b = 0..3 as
    //   low / high nibble of ql[64h + l] (b = 0 / 2) and of ql[64h + 32 + l] (b = 1 / 3), two more bits from
    //   qh[32h + l] >> 2b, scale scales[8h + 2b + l/16]                       (reference ggml-quants.c:1695-1711)
    // item x: p = x / 2 picks the ql half (k-blocks p and p + 2), hf = x & 1 the 16 values l = 16*hf + [0,16).
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        const int p = x >> 1, hf = x & 1;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            r.ql[h] = *reinterpret_cast<const u32x4_a2 *>(blk + 64 * h + 32 * p + 16 * hf);
            r.qh[h] = *reinterpret_cast<const u32x4_a2 *>(blk + 128 + 32 * h + 16 * hf);
        }
        r.sc = *reinterpret_cast<const u32x4_a2 *>(blk + 192);
        r.d = *reinterpret_cast<const unsigned short *>(blk + 208);
    }
    __device__ static __forceinline__ int kb0(int x) { return x >> 1; }
    __device__ static __forceinline__ int kb1(int x) { return (x >> 1) + 2; }
    // q: four 6-bit values 0..63 in bytes -> digits of q*sc + (4064 - 32*sc) = (q - 32)*sc + 4064 in 0..8160
    __device__ static __forceinline__ void digits(uint32_t q, uint32_t sc2, uint32_t bias2, uint32_t &hi, uint32_t &lo) {
        const uint32_t ev = q & 0x00ff00ffu, od = (q >> 8) & 0x00ff00ffu;
        const uint32_t ue = pk_mad16(ev, sc2, bias2), uo = pk_mad16(od, sc2, bias2);
        hi = ((ue >> 6) & 0x007f007fu) | (((uo >> 6) & 0x007f007fu) << 8);
        lo = (ue & 0x003f003fu) | ((uo & 0x003f003fu) << 8);
    }
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        const int p = x >> 1, hf = x & 1;
        // scales[8h + 2p + hf] and scales[8h + 2p + 4 + hf]: byte 2p + hf of dwords 2h and 2h + 1
        const int s0 = __builtin_amdgcn_sbfe((int)r.sc[2 * h], 8 * (2 * p + hf), 8);
        const int s1 = __builtin_amdgcn_sbfe((int)r.sc[2 * h + 1], 8 * (2 * p + hf), 8);
        const uint32_t sa = splat16((uint32_t)s0), ba = splat16((uint32_t)(Q6_BIAS - 32 * s0));
        const uint32_t sb = splat16((uint32_t)s1), bb = splat16((uint32_t)(Q6_BIAS - 32 * s1));
        const u32x4 ql = r.ql[h], qh = r.qh[h];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t hb = qh[i] >> (2 * p);
            const uint32_t q0 = (ql[i] & 0x0f0f0f0fu) | ((hb << 4) & 0x30303030u);            // k-block p
            const uint32_t q1 = ((ql[i] >> 4) & 0x0f0f0f0fu) | (hb & 0x30303030u);            // k-block p + 2
            uint32_t hi, lo;
            digits(q0, sa, ba, hi, lo);
            e.cell[0][0][i] = hi; e.cell[1][0][i] = lo;
            digits(q1, sb, bb, hi, lo);
            e.cell[0][1][i] = hi; e.cell[1][1][i] = lo;
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.d; }
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ float value(int p0, int p1, const float (&)[2], uint32_t dd, int corr) {
        return __builtin_fmaf(h2f(dd), (float)((p0 << 6) + p1 + corr), 0.f);
    }
};

template <> struct KQ<T_Q3_K> {
    static constexpr int BYTES = BYTES_Q3_K, NF16 = 0, NPL = 1;
    static constexpr bool HAS_BSUM = false, HALVES = false;
    // hmask[32] | qs[64] | scales[12] | d.  Element 128h + 32v + l: bits 2v of qs[32h + l], bit 4h + v of hmask[l], scale 8h + 2v + l/16.
    // Item x: the 16 bytes l = 16*(x & 1) + [0,16), k-blocks v = x / 2 and x / 2 + 2 (the two items of a k-half read the same bytes).
    struct Raw { u32x4 hm, q[2]; uint32_t s[3], d; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        const int hf = x & 1;
        r.hm = *reinterpret_cast<const u32x4_a2 *>(blk + 16 * hf);
        r.q[0] = *reinterpret_cast<const u32x4_a2 *>(blk + 32 + 16 * hf);
        r.q[1] = *reinterpret_cast<const u32x4_a2 *>(blk + 64 + 16 * hf);
#pragma unroll
        for (int i = 0; i < 3; i++) r.s[i] = *reinterpret_cast<const u32_a2 *>(blk + 96 + 4 * i);
        r.d = *reinterpret_cast<const unsigned short *>(blk + 108);
    }
    __device__ static __forceinline__ int kb0(int x) { return x >> 1; }
    __device__ static __forceinline__ int kb1(int x) { return (x >> 1) + 2; }
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        const int p = x >> 1, hf = x & 1;
        // 6-bit scale 4w + i is byte i of word w (reference ggml-quants.c:1062-1071): words 2h and 2h + 1 hold k-blocks 0, 1 and 2, 3
        const uint32_t hi2 = r.s[2] >> (4 * h);
        const uint32_t wa = ((r.s[0] >> (4 * h)) & 0x0f0f0f0fu) | ((hi2 & 0x03030303u) << 4);
        const uint32_t wb = ((r.s[1] >> (4 * h)) & 0x0f0f0f0fu) | (((hi2 >> 2) & 0x03030303u) << 4);
        const int b = 8 * (2 * p + hf);
        const int sc[2] = {(int)((wa >> b) & 0xffu) - 32, (int)((wb >> b) & 0xffu) - 32};
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int v = p + 2 * c;
            // byte = 128 + (4 - q)*sc in 0..252: the two bytes of a 16-bit lane never carry into each other, whatever the sign of
            // the multiplier (arithmetic modulo 2^16); flipping bit 7 gives the signed byte
            const uint32_t mul = splat16((uint32_t)(-sc[c])), add = splat16((uint32_t)((128 + 4 * sc[c]) * 0x101));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t q = ((r.q[h][i] >> (2 * v)) & 0x03030303u) | (((r.hm[i] >> (4 * h + v)) & 0x01010101u) << 2);
                e.cell[0][c][i] = pk_mad16(q, mul, add) ^ 0x80808080u;
            }
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.d; }
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ float value(int p0, int, const float (&)[2], uint32_t dd, int) {
        return __builtin_fmaf(h2f(dd), (float)-p0, 0.f);
    }
};

template <> struct KQ<T_Q2_K> {
    static constexpr int BYTES = BYTES_Q2_K, NF16 = 1, NPL = 1;    // fp16 product: sum_j m_j * bsum_j over the 16 sub-blocks
    static constexpr bool HAS_BSUM = false, HALVES = false;
    // scales[16] (low nibble scale, high nibble min) | qs[64] | d | dmin; quants, scales and items placed as in Q3_K
    struct Raw { u32x4 sc, q[2]; uint32_t dd; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        const int hf = x & 1;
        r.sc = *reinterpret_cast<const u32x4_a4 *>(blk);
        r.q[0] = *reinterpret_cast<const u32x4_a4 *>(blk + 16 + 16 * hf);
        r.q[1] = *reinterpret_cast<const u32x4_a4 *>(blk + 48 + 16 * hf);
        r.dd = *reinterpret_cast<const uint32_t *>(blk + 80);
    }
    __device__ static __forceinline__ int kb0(int x) { return x >> 1; }
    __device__ static __forceinline__ int kb1(int x) { return (x >> 1) + 2; }
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        const int p = x >> 1, b = 8 * (2 * p + (x & 1));
        const uint32_t s0 = splat16((r.sc[2 * h] >> b) & 15u), s1 = splat16((r.sc[2 * h + 1] >> b) & 15u);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            e.cell[0][0][i] = pk_mul16((r.q[h][i] >> (2 * p)) & 0x03030303u, s0);           // byte products <= 45
            e.cell[0][1][i] = pk_mul16((r.q[h][i] >> (2 * p + 4)) & 0x03030303u, s1);
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.dd; }
    // fp16 operand cell of item x < 2: mins of sub-blocks 8x .. 8x+7
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &r, int x) {
        u32x4 c;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = ((i < 2 ? r.sc[2 * (x & 1)] : r.sc[2 * (x & 1) + 1]) >> (16 * (i & 1) + 4)) & 0x0f0fu;
            c[i] = (uint32_t)__half_as_ushort(__float2half_rn((float)(w & 0xffu))) |
                   ((uint32_t)__half_as_ushort(__float2half_rn((float)(w >> 8))) << 16);    // exact
        }
        return c;
    }
    __device__ static __forceinline__ float value(int p0, int, const float (&f)[2], uint32_t dd, int) {
        return __builtin_fmaf(-h2f(dd >> 16), f[0], __builtin_fmaf(h2f(dd), (float)p0, 0.f));
    }
};

template <> struct KQ<T_IQ4_XS> {
    static constexpr int BYTES = BYTES_IQ4_XS, NF16 = 0, NPL = 2;
    static constexpr bool HAS_BSUM = true, HALVES = true;
    // d | u16 scales_h | scales_l[4] | qs[128]: sub-block ib is qs[16 ib ..], low nibbles elements 0..15, high nibbles 16..31.
    // Item x of stage h is sub-block 4h + x, both k-halves of k-block x.
    struct Raw { u32x2 h; u32x4 q[2]; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        r.h = *reinterpret_cast<const u32x2 *>(blk);
        r.q[0] = *reinterpret_cast<const u32x4_a4 *>(blk + 8 + 16 * x);
        r.q[1] = *reinterpret_cast<const u32x4_a4 *>(blk + 72 + 16 * x);
    }
    __device__ static __forceinline__ int kb0(int x) { return x; }
    __device__ static __forceinline__ int kb1(int x) { return x; }
    // four code indices (one per byte) -> code point + 128 of kvalues_iq4nl (reference ggml-common.h), 1..241
    __device__ static __forceinline__ uint32_t lookup4(uint32_t idx) {
        constexpr uint32_t F = 0x80808080u, T0 = 0xbfad9881u ^ F, T1 = 0xf6eaddcfu ^ F, T2 = 0x26190d01u ^ F, T3 = 0x71594535u ^ F;
        const uint32_t sel = idx & 0x07070707u;
        const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
        const uint32_t m = ((idx >> 3) & 0x01010101u) * 0xffu;
        return (lo & ~m) | (hi & m);
    }
    __device__ static __forceinline__ void emit(Emit &e, const Raw &r, int h, int x) {
        const int ib = 4 * h + x;
        const uint32_t nib = (r.h.y >> (4 * ib)) & 15u, top = (r.h.x >> (16 + 2 * ib)) & 3u;
        const int ls = (int)(nib | (top << 4)) - 32;
        const uint32_t mul = splat16((uint32_t)ls), bias = splat16((uint32_t)(Q6_BIAS - 128 * ls));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t hi, lo;
            KQ<T_Q6_K>::digits(lookup4(r.q[h][i] & 0x0f0f0f0fu), mul, bias, hi, lo);
            e.cell[0][0][i] = hi; e.cell[1][0][i] = lo;
            KQ<T_Q6_K>::digits(lookup4((r.q[h][i] >> 4) & 0x0f0f0f0fu), mul, bias, hi, lo);
            e.cell[0][1][i] = hi; e.cell[1][1][i] = lo;
        }
    }
    __device__ static __forceinline__ uint32_t scales(const Raw &r) { return r.h.x & 0xffffu; }
    __device__ static __forceinline__ u32x4 f16_cell(const Raw &, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ float value(int p0, int p1, const float (&)[2], uint32_t dd, int corr) {
        return __builtin_fmaf(h2f(dd), (float)((p0 << 6) + p1 + corr), 0.f);
    }
};

constexpr int KQ_PRODUCERS = 4;               // staging waves per workgroup, one per SIMD

template <int WT, int WR, int WC>
struct KqCfg {
    using T = KQ<WT>;
    static constexpr int NC = WR * WC;                             // MFMA waves
    static constexpr int NW = NC + KQ_PRODUCERS, NT = NW * 64;
    static constexpr int NPT = KQ_PRODUCERS * 64;                  // staging threads
    static constexpr int BM = 32 * WR;                             // weight rows per workgroup
    static constexpr int BN = 32 * KQ_TN * WC;                     // tokens per workgroup
    static constexpr int NF = T::NF16 > 0 ? T::NF16 : 1, NPL = T::NPL;
    // plane stride 2 mod 16 cells: the staging threads of one wave spread over the bank groups
    static constexpr int A_PLANE = BM + 2, B_PLANE = BN + 2;
    static constexpr int A_CELLS = NPL * KQ_KB * 2 * A_PLANE;   // 16-byte cells
    static constexpr int B_CELLS = KQ_KB * 2 * B_PLANE;
    // one stage buffer (two of them, by stage parity)
    static constexpr size_t OFF_A = 0;
    static constexpr size_t OFF_B = OFF_A + (size_t)A_CELLS * 16;
    static constexpr size_t STAGE = OFF_B + (size_t)B_CELLS * 16;
    // one super-block buffer (two of them, by super-block parity)
    static constexpr size_t OFF_FA = 0;                                     // fp16 cells [NF16][k-half][BM]: m_j (sc_j) twice
    static constexpr size_t OFF_FB = OFF_FA + (size_t)NF * 2 * BM * 16;     // fp16 cells [k-half][BN]: the token's 16 bsums
    static constexpr size_t OFF_SD = OFF_FB + (size_t)2 * BN * 16;          // u32 [BM]: d | dmin << 16, permuted per 32 rows
    static constexpr size_t OFF_SX = OFF_SD + (size_t)BM * 4;               // f32 [BN]: activation scale of the super-block
    static constexpr size_t OFF_SC = OFF_SX + (size_t)BN * 4;               // i32 [BN]: -4064 * sum of the token's quants
    static constexpr size_t SBLK = OFF_SC + (size_t)BN * 4;
    static constexpr size_t OFF_STAGES = 0;
    static constexpr size_t OFF_SBLK = 2 * STAGE;
    static constexpr size_t OFF_DUMP = OFF_SBLK + 2 * SBLK;                 // 16 bytes per staging thread: where stores that do not apply go
    static constexpr size_t TOTAL = OFF_DUMP + (size_t)NPT * 16;
    static constexpr int W_ITEMS = BM * 4;
    static constexpr int W_PER_T = W_ITEMS / NPT;
    static constexpr int X_ITEMS = BN * KQ_KB * 2;
    static constexpr int X_PER_T = X_ITEMS / NPT;
    static_assert(2 * BN <= NPT, "two staging threads per token convert its block sums");
    static_assert(W_ITEMS % NPT == 0 && X_ITEMS % NPT == 0, "staging items divide evenly over the staging threads");
    static_assert(STAGE % 16 == 0 && SBLK % 16 == 0, "buffers keep 16-byte alignment");
};

// A workgroup is WR x WC MFMA waves plus four staging waves (one per SIMD).  Per stage (4 k-blocks = half a
// super-block; LDS double buffered; one barrier per stage):
//
//     staging waves : global loads of stage s+3 | expand stage s+1 (loaded two stages ago) into the other buffer
//     MFMA waves    : 4 k-blocks of MFMAs from the current buffer | after a super-block's second half: fold
//
// The two kinds of wave run side by side on every SIMD, so operand expansion (vector pipe, LDS writes, memory
// latency) overlaps the matrix pipe by construction instead of by instruction scheduling.  Nothing in the loops is
// conditional: loads past the last stage repeat it, and stores that do not apply go to a per-thread dump slot.
template <int WT, int WR, int WC, int OCC, bool GATHER>
__global__ __launch_bounds__((WR * WC + KQ_PRODUCERS) * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void gemm_kq_kernel(const uint8_t *__restrict__ W, size_t nb01, int64_t K, int64_t N, const uint8_t *__restrict__ ws,
                    size_t ws_stride, int64_t M, float *__restrict__ y, int64_t ldy, TileMap map, RowGather rg, int slice_sb) {
    using T = KQ<WT>;
    using C = KqCfg<WT, WR, WC>;
    constexpr int TN = KQ_TN;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // split K (never with a gather, whose grid rows are the experts): grid row s takes super-blocks sb0 .. of every row
    // and writes its partial tile to slice s of y
    int sb0 = 0, nstages = (int)(K / QK_K) * 2;
    if (!GATHER && slice_sb > 0) {
        sb0 = (int)blockIdx.y * slice_sb;
        nstages = 2 * min(slice_sb, (int)(K / QK_K) - sb0);
        y += (size_t)blockIdx.y * (size_t)M * (size_t)ldy;
    }
    const TileCoord tc = xcd_tile(blockIdx.x, map);
    if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;        // padding of the tile map
    size_t w_offset;
    const GatherView gv = resolve_gather<GATHER>(rg, w_offset, M);                   // MUL_MAT_ID: this expert's rows
    W += w_offset;
    const int64_t row_base = (int64_t)tc.row_tile * C::BM;
    if (gv.tok_tile < 0) return;
    const int64_t tok_base = (int64_t)(GATHER ? gv.tok_tile : tc.tok_tile) * C::BN;
    if (tok_base >= M) return;

    if (wave >= C::NC) {
        // ------------------------------------------------------------------------------------ staging waves
        const int pt = tid - C::NC * 64;
        const size_t off_d = q8_K_off_d(K), off_bs = q8_K_off_bsums(K);
        uint8_t *const dump = lds + C::OFF_DUMP + pt * 16;
        struct Acts {
            u32x4 x[C::X_PER_T];
            u32x4 bs;          // 8 of the token's bsums (threads 2*token + k-half)
            float xs;
            int xc;
        };
        struct Wts { typename T::Raw w[C::W_PER_T]; };
        Acts E, O;             // activations of an even / odd stage
        Wts W0, W1;            // weights of an even / odd super-block (both halves: every cache line is fetched once)
        // per-thread source addresses of stage 0 (they advance by a constant per stage / super-block)
        const uint8_t *wsrc[C::W_PER_T], *xsrc[C::X_PER_T];
#pragma unroll
        for (int i = 0; i < C::W_PER_T; i++) wsrc[i] = W + (size_t)min(row_base + ((pt + i * C::NPT) >> 2), N - 1) * nb01;
#pragma unroll
        for (int i = 0; i < C::X_PER_T; i++)
            xsrc[i] = ws + (size_t)gv.act_row(min(tok_base + ((pt + i * C::NPT) >> 3), M - 1)) * ws_stride + 16 * ((pt + i * C::NPT) & 7);
        // activation scale: thread t < BN for token t; block sums: thread t < 2*BN for token t/2, half t&1
        const uint8_t *ssrc = ws + (size_t)gv.act_row(min(tok_base + min(pt, C::BN - 1), M - 1)) * ws_stride;
        const uint8_t *bsrc = ws + (size_t)gv.act_row(min(tok_base + min(pt >> 1, C::BN - 1), M - 1)) * ws_stride + off_bs + 16 * (pt & 1);
        const int nsb = nstages >> 1;

        auto fetch_w = [&](Wts &R, int sb_wanted) {
            const int sb = min(sb_wanted, nsb - 1);
#pragma unroll
            for (int i = 0; i < C::W_PER_T; i++) T::fetch(R.w[i], wsrc[i] + (size_t)(sb0 + sb) * T::BYTES, (pt + i * C::NPT) & 3);
        };
        auto fetch_x = [&](Acts &R, int stage_wanted, auto even_tag) {
            constexpr bool even = decltype(even_tag)::value;
            const int stage = min(stage_wanted, nstages - 1);
            const int sb = stage >> 1;
#pragma unroll
            for (int i = 0; i < C::X_PER_T; i++) R.x[i] = *reinterpret_cast<const u32x4 *>(xsrc[i] + (size_t)(2 * sb0 + stage) * (32 * KQ_KB));
            if constexpr (even) {
                R.xs = reinterpret_cast<const float *>(ssrc + off_d)[sb0 + sb];
                if constexpr (T::NF16 > 0) R.bs = *reinterpret_cast<const u32x4 *>(bsrc + (size_t)(sb0 + sb) * 32);
                if constexpr (T::HAS_BSUM) {
                    const u32x4 *bp = reinterpret_cast<const u32x4 *>(ssrc + off_bs + (size_t)(sb0 + sb) * 32);
                    const u32x4 b0 = bp[0], b1 = bp[1];
                    const uint32_t w[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
                    int sum = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++) sum += (int)(int16_t)(w[j] & 0xffffu) + ((int)w[j] >> 16);
                    R.xc = -Q6_BIAS * sum;
                }
            }
        };

        // expand a prefetched stage into LDS buffer `buf`; even stages also carry the super-block's scales
        auto commit = [&](const Wts &RW, const Acts &R, int buf, int sbp, auto even_tag) {
            constexpr bool even = decltype(even_tag)::value;
            constexpr int h = even ? 0 : 1;
            uint8_t *base = lds + C::OFF_STAGES + (size_t)buf * C::STAGE;
            uint8_t *sblk = lds + C::OFF_SBLK + (size_t)sbp * C::SBLK;
            u32x4 *A = reinterpret_cast<u32x4 *>(base + C::OFF_A);
            u32x4 *B = reinterpret_cast<u32x4 *>(base + C::OFF_B);
#pragma unroll
            for (int i = 0; i < C::W_PER_T; i++) {
                const int item = pt + i * C::NPT;
                const int r = item >> 2, x = item & 3;
                Emit e;
                T::emit(e, RW.w[i], h, x);
                const int c0 = cell_pos<T>(x, 0), c1 = cell_pos<T>(x, 1);
#pragma unroll
                for (int pl = 0; pl < C::NPL; pl++) {
                    A[(pl * KQ_KB * 2 + c0) * C::A_PLANE + r] = e.cell[pl][0];
                    A[(pl * KQ_KB * 2 + c1) * C::A_PLANE + r] = e.cell[pl][1];
                }
                if constexpr (even) {
                    // the lane that owns MFMA result register v of a 32-row tile holds row 8*(v/4) + 4*half + v%4:
                    // keep the scale of row i at half*16 + (i/8)*4 + i%4 so a lane reads its 16 scales contiguously
                    const int i32 = r & 31;
                    const int pos = ((i32 >> 2) & 1) * 16 + (i32 >> 3) * 4 + (i32 & 3);
                    uint8_t *dst = (x == 0) ? sblk + C::OFF_SD + ((r & ~31) + pos) * 4 : dump;
                    *reinterpret_cast<uint32_t *>(dst) = T::scales(RW.w[i]);
                    if constexpr (T::NF16 > 0) {
                        // items x < 2*NF16 of a row each build one fp16 operand cell [x/2][x&1][row]
                        uint8_t *fd = (x < 2 * T::NF16) ? sblk + C::OFF_FA + (size_t)(x * C::BM + r) * 16 : dump;
                        *reinterpret_cast<u32x4 *>(fd) = T::f16_cell(RW.w[i], x);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < C::X_PER_T; i++) {
                const int item = pt + i * C::NPT;
                B[(item & 7) * C::B_PLANE + (item >> 3)] = R.x[i];
            }
            if constexpr (even) {
                uint8_t *dx = (pt < C::BN) ? sblk + C::OFF_SX + pt * 4 : dump;
                *reinterpret_cast<float *>(dx) = R.xs;
                if constexpr (T::HAS_BSUM) {
                    uint8_t *dc = (pt < C::BN) ? sblk + C::OFF_SC + pt * 4 : dump;
                    *reinterpret_cast<int *>(dc) = R.xc;
                }
                if constexpr (T::NF16 > 0) {
                    uint8_t *fb = (pt < 2 * C::BN) ? sblk + C::OFF_FB + (size_t)((pt & 1) * C::BN + (pt >> 1)) * 16 : dump;
                    *reinterpret_cast<u32x4 *>(fb) = i16x8_to_f16(R.bs);
                }
            }
        };

        // the two staging steps that run while the MFMA waves work on super-block j (weights in `cur`); `nxt` holds
        // super-block j + 1, and `cur` is refilled with super-block j + 2 once its second half has been expanded
        auto steps = [&](Wts &cur, Wts &nxt, int j) {
            fetch_x(E, 2 * j + 2, std::true_type{});
            commit(cur, O, 1, j & 1, std::false_type{});                  // stage 2j + 1, during stage 2j
            __syncthreads();
            fetch_x(O, 2 * j + 3, std::false_type{});
            fetch_w(cur, j + 2);
            commit(nxt, E, 0, (j + 1) & 1, std::true_type{});             // stage 2j + 2, during stage 2j + 1 and the fold
            __syncthreads();
        };

        fetch_w(W0, 0);
        fetch_x(E, 0, std::true_type{});
        fetch_x(O, 1, std::false_type{});
        fetch_w(W1, 1);
        commit(W0, E, 0, 0, std::true_type{});
        __syncthreads();
        for (int j = 0; j < nsb; j += 2) {
            steps(W0, W1, j);
            if (j + 1 < nsb) steps(W1, W0, j + 1);
        }
        return;
    }

    // ------------------------------------------------------------------------------------------ MFMA waves
    const int wr = wave / WC, wc = wave % WC;
    const int half = lane >> 5, l32 = lane & 31;
    const int r0 = wr * 32, n0 = wc * TN * 32;

    i32x16 P[C::NPL][TN];
    float out[TN][16];
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
        for (int v = 0; v < 16; v++) out[c][v] = 0.f;

    // 4 k-blocks of one stage; `first` starts the super-block's accumulators from zero
    auto compute = [&](int buf, auto first_tag) {
        constexpr bool first = decltype(first_tag)::value;
        const uint8_t *base = lds + C::OFF_STAGES + (size_t)buf * C::STAGE;
        const u32x4 *A = reinterpret_cast<const u32x4 *>(base + C::OFF_A);
        const u32x4 *B = reinterpret_cast<const u32x4 *>(base + C::OFF_B);
#pragma unroll
        for (int b = 0; b < KQ_KB; b++) {
            i32x4 af[C::NPL], bf[TN];
#pragma unroll
            for (int pl = 0; pl < C::NPL; pl++) {
                const u32x4 t = A[((pl * KQ_KB + b) * 2 + half) * C::A_PLANE + r0 + l32];
                af[pl] = i32x4{(int)t.x, (int)t.y, (int)t.z, (int)t.w};
            }
#pragma unroll
            for (int c = 0; c < TN; c++) {
                const u32x4 t = B[(b * 2 + half) * C::B_PLANE + n0 + c * 32 + l32];
                bf[c] = i32x4{(int)t.x, (int)t.y, (int)t.z, (int)t.w};
            }
#pragma unroll
            for (int pl = 0; pl < C::NPL; pl++)
#pragma unroll
                for (int c = 0; c < TN; c++) {
                    if (first && b == 0) {
                        const i32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                        P[pl][c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[pl], bf[c], zero, 0, 0, 0);
                    } else {
                        P[pl][c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[pl], bf[c], P[pl][c], 0, 0, 0);
                    }
                }
        }
    };

    // once per super-block: the fp16 products against the block sums, then fold the planes and apply d, dmin and
    // the activation scale
    auto fold = [&](int sbp) {
        const uint8_t *sblk = lds + C::OFF_SBLK + (size_t)sbp * C::SBLK;
        const u32x4 *sp = reinterpret_cast<const u32x4 *>(sblk + C::OFF_SD) + (r0 + half * 16) / 4;
        const u32x4 s0 = sp[0], s1 = sp[1], s2 = sp[2], s3 = sp[3];
        const uint32_t sd[16] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w, s2.x, s2.y, s2.z, s2.w, s3.x, s3.y, s3.z, s3.w};
        f16x8 fa[C::NF];
        if constexpr (T::NF16 > 0) {
#pragma unroll
            for (int f = 0; f < T::NF16; f++)
                fa[f] = *reinterpret_cast<const f16x8 *>(sblk + C::OFF_FA + (size_t)((2 * f + half) * C::BM + r0 + l32) * 16);
        }
#pragma unroll
        for (int c = 0; c < TN; c++) {
            f32x16 F[2];
            if constexpr (T::NF16 > 0) {
                const f16x8 fb = *reinterpret_cast<const f16x8 *>(sblk + C::OFF_FB + (size_t)(half * C::BN + n0 + c * 32 + l32) * 16);
                const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int f = 0; f < T::NF16; f++) F[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[f], fb, zero, 0, 0, 0);
            }
            const float dx = reinterpret_cast<const float *>(sblk + C::OFF_SX)[n0 + c * 32 + l32];
            int corr = 0;
            if constexpr (T::HAS_BSUM) corr = reinterpret_cast<const int *>(sblk + C::OFF_SC)[n0 + c * 32 + l32];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                float f[2] = {0.f, 0.f};
#pragma unroll
                for (int j = 0; j < T::NF16; j++) f[j] = F[j][v];
                out[c][v] = __builtin_fmaf(T::value(P[0][c][v], P[C::NPL - 1][c][v], f, sd[v], corr), dx, out[c][v]);
            }
        }
    };

    __syncthreads();                                                    // stage 0 is in LDS
    for (int s = 0; s < nstages; s += 2) {
        compute(0, std::true_type{});
        __syncthreads();
        compute(1, std::false_type{});
        fold((s >> 1) & 1);
        __syncthreads();
    }

    // ---- epilogue: register v of token tile c is row 8*(v/4) + 4*half + v%4, token l32 ----
#pragma unroll
    for (int c = 0; c < TN; c++) {
        const int64_t tok = tok_base + n0 + c * 32 + l32;
        if (tok >= M) continue;
        const int64_t orow = gv.out_row(tok);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int64_t row = row_base + r0 + 8 * g + 4 * half;
            float *dst = y + (size_t)orow * ldy + row;
            if (row + 3 < N && (((uintptr_t)dst) & 15) == 0) {
                *reinterpret_cast<float4 *>(dst) = make_float4(out[c][4 * g], out[c][4 * g + 1], out[c][4 * g + 2], out[c][4 * g + 3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (row + e < N) dst[e] = out[c][4 * g + e];
            }
        }
    }
}

static bool kq_splittable(int64_t N) { return ceil_div(N, (int64_t)64) <= 128; }
// How gemm_kr_kernel covers a product with `tiles` of 128 rows x 64 tokens: k groups of a workgroup (1: four waves, two workgroups
// a CU; 2: eight waves, one workgroup a CU) and slices of K over the grid's second dimension.
//   more tiles than CUs     one group: two independent workgroups a CU (us, 512 tokens x 4096 values, one / two groups: Q4_K 4608 rows
//                           48 / 55, 14336 rows 93 / 112; Q6_K 62 / 76, 120 / 142)
//   above half as many      two groups walk the super-blocks in turn, so that every SIMD has two waves (4096 rows: Q4_K 37.5 / 33.7,
//                           Q5_K 40 / 38.5, Q2_K 29 / 27; Q3_K 31.8 / 30.5); so too with 2 slices of rows above 8192 values
//                           (14336 values x 4096 rows at 201 tokens: Q4_K 59 / 54, Q3_K 53 / 48)
//   fewer                   as many slices as give every CU a workgroup, at most 8, or 16 of four super-blocks (a slice more costs its
//                           partial outputs: Q4_K 14336 values x 4096 rows at 64 tokens 88, 53, 34, 27, 30 us in 1, 2, 4, 8, 12; 1024
//                           rows at 17 tokens 18.0 / 16.6 in 8 / 12).  Not rounded up: 96 tiles in 3 slices leave 32 workgroups for a
//                           second turn (Q6_K 4096 x 4096 at 130 tokens 29 / 31 us in 2 / 3).  The slice sum pays for at most
//                           150000 partial outputs a super-block of a row (1024 values x 4096 rows whole / in 4: Q4_K 17 tokens 12.5 /
//                           11.6, Q3_K 64 tokens 12.8 / 13.3; 1792 x 4096 at 64 tokens 19 / 16), not for rows of three or less or for two slices of less than 8.
struct KrPlan { int groups, slices; };
static KrPlan kr_plan(int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int64_t tiles = ceil_div(N, (int64_t)128) * ceil_div(M, (int64_t)64), units = K / QK_K;
    if (tiles > cus || units == 1) return KrPlan{1, 1};
    const int64_t most = std::max<int64_t>(8, std::min<int64_t>(16, units / 4));
    int64_t s = units < 4 ? 1 : std::min({cus / tiles, units, most, units * 150000 / (M * N)});
    if (s < (units < 8 ? 3 : 2)) return KrPlan{units < 4 ? 1 : 2, 1};
    const int64_t per = ceil_div(units, s);
    s = ceil_div(units, per);                                           // no empty slice
    return KrPlan{s == 2 && units > 32 ? 2 : 1, (int)s};
}
// Q6_K with a tile for at most every CU and more than a third as many: gemm_kq_kernel, whose staging waves expand a weight once for
// 128 tokens, in slices of its own (us, staged / gemm_kr_kernel: 14336 values x 4096 rows at 512 tokens 115 / 121, 250 tokens 69 / 72, 130
// tokens 66 / 69; 4096 x 4096 at 250 tokens 31 / 32, 512 tokens 42 / 41.5).
static bool kq_staged(int wtype, int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int64_t tiles = ceil_div(N, (int64_t)128) * ceil_div(M, (int64_t)64);
    if (wtype != T_Q6_K || tiles > cus) return false;
    return K < 8 * QK_K || (3 * tiles > cus && (M > 128 || kq_splittable(N)));
}
// Its slices of K for 64 x 128 tiles: up to two workgroups per CU with one token tile, one per CU with more, at least four super-blocks
// each.  low_bit_gemm_ahead below was fitted to times of that kernel and asks for them too.
static int kq_staged_slices(int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int64_t units = K / QK_K, tiles = ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)128);
    if (units < 8 || (M <= 128 && !kq_splittable(N))) return 1;
    const int64_t s = std::min({(M <= 128 ? 2 : 1) * cus / tiles, units / 4, (int64_t)16});
    if (s < 2) return 1;
    const int64_t per = ceil_div(units, s);
    return (int)ceil_div(units, per);
}
static int planned_slices(int wtype, int64_t K, int64_t N, int64_t n, int64_t cus) {
    return kq_staged(wtype, K, N, n, cus) ? kq_staged_slices(K, N, n, cus) : kr_plan(K, N, n, cus).slices;
}
// With few tokens the GEMM's time is its walk over K, whatever the token count, while the GEMV forms pass over the weights once
// per 8 (Q6_K) or 16 tokens (Q4_K, Q5_K) at memory speed.  The GEMM as planned above is ahead from the first token of a second pass on
// (us, GEMV passes / GEMM: Q4_K at 17 tokens 4096 x 4096 17.4 / 14.3, 1024 values x 2048 rows 17.9 / 11.0, 4096 values x 16640 rows at 20 tokens
// 35 / 27; Q6_K at 17 tokens 1280 x 8192 34 / 16).  Where it wants slices and the caller's workspace has no room for their partial
// outputs, the unsplit walk pays later.
static int64_t gemm_kq_min_tokens(int wtype, int64_t K, int64_t N, int64_t n, bool can_split) {
    if (can_split || planned_slices(wtype, K, N, n, 256) == 1) return wtype == T_Q6_K ? 9 : 17;
    const bool long_rows = K > 8192;
    return wtype == T_Q6_K ? (long_rows ? 41 : 25) : (long_rows ? 33 : 49);
}

// Q3_K, Q2_K and IQ4_XS: the dot-product GEMV passes of 8 tokens, whose time grows with the tokens, against the GEMM, whose time
// below 128 tokens does not.  A token count alone does not part them (GEMV / GEMM, us, split K: IQ4_XS 8192 x 8192 at 12
// tokens 36 / 43, 1024 x 14336 at 9 tokens 20 / 19; Q2_K 1024 x 4096 at 10 tokens 12 / 14, 4096 x 4096 at 9 tokens 16 / 15;
// unsplit: IQ4_XS 748 x 7168 at 32 tokens 34 / 58, 4096 x 1024 at 25 tokens 32 / 14), so both times are estimated, in us, with terms
// fitted to 5000 measured products (to 13 and 9 per cent for nine in ten of them):
//   GEMV   a launch per pass, then per token the rounds of 1024 rows (four a CU) and of 4096 values of a row
//   GEMM   quantizer and launch (and slice sum), then the super-blocks a workgroup walks times the rounds of 256 workgroups; split K
//          has most of the weights in flight at once and pays for their bytes too
static bool low_bit_gemm_ahead(int wtype, int64_t K, int64_t N, int64_t n, int slices) {
    if (n < 9) return false;                                         // one GEMV pass
    const int64_t group = gemv_max_tokens(wtype, K, DeviceLimits{256, 160 * 1024});      // 8, fewer on very long rows
    if (group < 1) return true;
    const float passes = (float)ceil_div(n, group), rows = (float)ceil_div(N, (int64_t)1024), parts = (float)ceil_div(K, (int64_t)4096);
    const float gemv = passes * (4.6f + 0.235f * rows) + (float)n * parts * (0.135f + 0.103f * rows);
    const int64_t tiles = ceil_div(N, (int64_t)64) * ceil_div(n, (int64_t)128) * slices;
    const float walk = (wtype == T_Q3_K ? 1.12f : wtype == T_Q2_K ? 1.23f : 1.84f) * (float)ceil_div(K / QK_K, (int64_t)slices) *
                       (float)ceil_div(tiles, (int64_t)256);
    const float gemm = slices == 1 ? 7.1f + walk : 9.2f + 0.82f * walk + 0.14f * (float)N * (float)K / 1048576.f;
    return gemm < gemv;
}
bool gemm_kq_type(int wtype) {
    return wtype == T_Q4_K || wtype == T_Q5_K || wtype == T_Q6_K || wtype == T_Q3_K || wtype == T_Q2_K || wtype == T_IQ4_XS;
}
bool gemm_kq_supported(int wtype, int64_t K, int64_t N, int64_t n, bool can_split) {
    if (!gemm_kq_type(wtype) || K < QK_K || K % QK_K != 0 || N < 1) return false;
    const int64_t forced = tune("CHIP_GEMM_MIN_TOKENS", 0);
    if (forced > 0) return n >= forced;
    if (wtype == T_Q3_K || wtype == T_Q2_K || wtype == T_IQ4_XS)
        return low_bit_gemm_ahead(wtype, K, N, n, can_split ? kq_staged_slices(K, N, n, 256) : 1);
    return n >= gemm_kq_min_tokens(wtype, K, N, n, can_split);
}
int gemm_kq_slices(int wtype, int64_t K, int64_t N, int64_t n, int compute_units) {
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    if (!gemm_kq_supported(wtype, K, N, n, true)) return 1;
    return planned_slices(wtype, K, N, n, cus);
}

template <int WT, int WR, int WC, int OCC, bool GATHER>
static hipError_t launch_kq(const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride, int64_t M,
                            float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather &rg, int64_t n_as,
                            int slices = 1, float *part = nullptr) {
    using C = KqCfg<WT, WR, WC>;
    const size_t lds_bytes = C::TOTAL;
    if ((int64_t)lds_bytes > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kq_kernel<WT, WR, WC, OCC, GATHER>;
    static LdsGrant grant;                                               // one per kernel instantiation
    if (hipError_t e = grant_dynamic_lds(kfn, lds_bytes, lim, grant); e != hipSuccess) return e;
    // one workgroup per CU: 32 workgroups run on an XCD at a time
    const TileMap map = make_tile_map(ceil_div(N, C::BM), GATHER ? 1 : ceil_div(M, C::BN), 32);
    if (!GATHER && slices > 1) {
        const int slice_sb = (int)ceil_div(K / QK_K, (int64_t)slices);
        hipLaunchKernelGGL(kfn, dim3(map.grid, (unsigned)slices), dim3(C::NT), lds_bytes, st, (const uint8_t *)W, nb01, K, N,
                           (const uint8_t *)ws, ws_stride, M, part, N, map, rg, slice_sb);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        return launch_sum_slices(part, slices, M, N, y, ldy, st);
    }
    hipLaunchKernelGGL(kfn, dim3(map.grid, (unsigned)n_as), dim3(C::NT), lds_bytes, st, (const uint8_t *)W, nb01, K, N,
                       (const uint8_t *)ws, ws_stride, M, y, ldy, map, rg, 0);
    return hipGetLastError();
}

template <int WT>
static hipError_t launch_kq_type(const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride,
                                 int64_t M, float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather &rg,
                                 int64_t n_as, SplitK split) {
    if (rg.perm)                                                                     // expert groups: 64 x 128 tiles
        return launch_kq<WT, 2, 2, 2, true>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as);
    const int64_t cus = lim.compute_units > 0 ? lim.compute_units : 256;
    auto room = [&](int slices) {
        return slices <= 1 || (split.part && split.bytes >= (size_t)slices * (size_t)M * (size_t)N * sizeof(float) && (((uintptr_t)split.part) & 15) == 0);
    };
    KrPlan p = kr_plan(K, N, M, cus);
    if constexpr (WT == T_Q6_K) {
        const bool staged = kq_staged(WT, K, N, M, cus);
        if (staged || !room(p.slices)) {                                             // (the unsplit walk of few tiles: staged too)
            const int slices = staged ? kq_staged_slices(K, N, M, cus) : 1;
            return launch_kq<WT, 2, 2, 2, false>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, room(slices) ? slices : 1, split.part);
        }
    }
    if (!room(p.slices)) p = KrPlan{2, 1};
    return launch_gemm_kr(p.groups, WT, W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, p.slices, split.part);
}

// MUL_MAT_ID of Q3_K, Q2_K and IQ4_XS, both times estimated in us as above.  A GEMV per (token, expert) pair costs its rows by
// the 4096 values; the GEMM walks a whole 64 x 128 tile per row tile of a picked expert, for a single pair too, and an XCD (32 CUs)
// runs one in eight of an expert's row tiles.  With ids drawn evenly n_as * (1 - e^(-pairs / n_as)) experts are picked.
// (GEMV / GEMM, us: Q2_K 768 x 2048, 128 experts, 64 pairs 18 / 53, 1024 pairs 194 / 119; Q3_K 2048 x 768 at 256 pairs 171 / 87;
// 14336 x 4096, 8 experts, 64 pairs 294 / 166.  Of 1500 drawn calls 12 took the
// slower kernel by more than 5 %, the worst by 28 %: Q3_K 2048 x 768, 128 experts, 64 pairs 47 / 60.)
bool gemm_kq_moe_ahead(int wtype, int64_t K, int64_t N, int64_t n_as, int64_t pairs) {
    if (wtype != T_Q3_K && wtype != T_Q2_K && wtype != T_IQ4_XS) return true;
    if (gemv_max_tokens(wtype, K, DeviceLimits{256, 160 * 1024}) < 1) return true;
    const float n_pairs = (float)pairs, experts = (float)n_as;
    const float gemv = 7.5f + (wtype == T_Q3_K ? 0.34f : wtype == T_Q2_K ? 0.238f : 0.382f) * n_pairs * (float)N / 1024.f * (float)ceil_div(K, (int64_t)4096);
    const float per_sb = wtype == T_Q3_K ? 0.95f : wtype == T_Q2_K ? 1.05f : 1.6f;
    const float tiles = experts * (1.f - std::exp(-n_pairs / experts)) + n_pairs / 128.f;
    const float rounds = (float)ceil_div(ceil_div(N, (int64_t)64), (int64_t)8) * tiles / 32.f + 0.3f;
    const float gemm = 12.f + (rounds > 1.f ? rounds : 1.f) * (per_sb * (float)(K / QK_K) + 2.2f);
    return gemm < gemv;
}
int gemm_kq_moe_tile_tokens() { return KqCfg<T_Q4_K, 2, 2>::BN; }      // the 64 x 128 shape serves the expert groups

hipError_t launch_gemm_kq(int wtype, const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride,
                          int64_t M, float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather *rgp, int64_t n_as,
                          SplitK split) {
    if (M <= 0 || N <= 0 || n_as <= 0) return hipSuccess;
    const RowGather rg = rgp ? *rgp : RowGather{nullptr, nullptr, nullptr, 1, 1, 0};
    switch (wtype) {
        case T_Q4_K: return launch_kq_type<T_Q4_K>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        case T_Q5_K: return launch_kq_type<T_Q5_K>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        case T_Q6_K: return launch_kq_type<T_Q6_K>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        case T_Q3_K: return launch_kq_type<T_Q3_K>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        case T_Q2_K: return launch_kq_type<T_Q2_K>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        case T_IQ4_XS: return launch_kq_type<T_IQ4_XS>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, split);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace chip
