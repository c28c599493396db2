// Per K-quant type: where a lane's 16 values of a super-block lie and how they become int8 MFMA operands.  Of the two GEMMs whose waves expand
// their own rows (gemm_kquant_rows.hip, which says what the digit planes are, and gemm_kquant_few.hip).
#pragma once
#include "kquant_dev.h"

namespace chip {
namespace {

// 6-bit scales and mins of sub-blocks 2jp and 2jp+1 (low byte, next byte) from the 12 packed bytes that follow
// d and dmin (reference ggml-quants.c:625-632)
__device__ __forceinline__ void scale_min_pair(const u32x4 &h, int jp, uint32_t &sc, uint32_t &mn) {
    const int sh = 16 * (jp & 1);
    const uint32_t a1 = h.y >> sh, a2 = h.z >> sh, a3 = h.w >> sh;
    if (jp < 2) { sc = a1 & 0x3f3fu; mn = a2 & 0x3f3fu; }
    else        { sc = (a3 & 0x0f0f0f0fu & 0xffffu) | ((a1 >> 2) & 0x3030u); mn = ((a3 >> 4) & 0x0f0fu) | ((a2 >> 2) & 0x3030u); }
}
// the same for four sub-blocks at once, one per byte: sub-blocks 0..3 (g = 0) or 4..7 (g = 1)
__device__ __forceinline__ void scale_min_quad(const u32x4 &h, int g, uint32_t &sc, uint32_t &mn) {
    const uint32_t sc0 = h.y & 0x3f3f3f3fu, mn0 = h.z & 0x3f3f3f3fu;
    const uint32_t sc1 = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u), mn1 = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    sc = g ? sc1 : sc0;
    mn = g ? mn1 : mn0;
}
// two small integers -> fp16 (exact)
__device__ __forceinline__ uint32_t f16_pair(uint32_t a, uint32_t b) {
    return (uint32_t)__half_as_ushort(__float2half_rn((float)a)) | ((uint32_t)__half_as_ushort(__float2half_rn((float)b)) << 16);
}
// four small integers (one per byte) -> the fp16 operand cell {b0, b0, b1, b1, b2, b2, b3, b3}: sub-block j stands
// against the two 16-value bsums 2j and 2j+1
__device__ __forceinline__ u32x4 bytes_to_f16_pairs(uint32_t v) {
    u32x4 c;
#pragma unroll
    for (int i = 0; i < 4; i++) c[i] = f16_pair((v >> (8 * i)) & 0xffu, (v >> (8 * i)) & 0xffu);
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
__device__ __forceinline__ float mul_add(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double mul_add(double a, double b, double c) { return __builtin_fma(a, b, c); }
// Per weight type.  A super-block is fetched as NCH 16-byte chunks (the last one ends with the super-block, so it may overlap the
// one before) and kept in LDS in that order, NCH cells a row.  Where NCH is odd, 16 rows' cells of one index fall into different banks; for Q6_K (14
// cells) and Q2_K (6) two of them share one.
// A lane reads its share back: hdr() what all items need, load() the 16-value k-half hf of the two k-blocks of item (H, p), NEXT apart in half H of
// the super-block (kr_k_block), which expand() turns into MFMA operand cells [k-block][plane].  H is known at compile time; p and hf may be the lane's.
// value() is the super-block's d * sumi - dmin * summ, in 32 or in 64 bits.
template <int WT> struct KR;

template <> struct KR<T_Q4_K> {
    static constexpr int BYTES = BYTES_Q4_K, NCH = 9, NPL = 2, NF16 = 1;
    typedef u32x4 chunk_t;
    struct Hdr { u32x4 h; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int) { return Hdr{row[0]}; }
    static constexpr int NEXT = 1;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int hf) { return Raw{row[1 + 4 * H + 2 * p + hf]}; }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int, u32x4 (&c)[2][2]) {
        uint32_t sc, mn;
        scale_min_pair(h.h, 2 * H + p, sc, mn);
        const uint32_t sh0 = (sc >> 3) & 7u, sl0 = sc & 7u, sh1 = sc >> 11, sl1 = (sc >> 8) & 7u;
        const u32x4 q = r.q;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = q[i] & 0x0f0f0f0fu, hi = (q[i] >> 4) & 0x0f0f0f0fu;
            c[0][0][i] = lo * sh0; c[0][1][i] = lo * sl0;                             // four byte products <= 105: no carries
            c[1][0][i] = hi * sh1; c[1][1][i] = hi * sl1;
        }
    }
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &h, int, int half) {
        uint32_t sc, mn;
        scale_min_quad(h.h, half, sc, mn);
        return bytes_to_f16_pairs(mn);
    }
    __device__ static __forceinline__ u32x2 f16_quad(const u32x4 *row, int g) {           // against the block sums 4g .. 4g + 3
        uint32_t sc, mn;
        scale_min_pair(row[0], g, sc, mn);
        return u32x2{f16_pair(mn & 0xffu, mn & 0xffu), f16_pair(mn >> 8, mn >> 8)};
    }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.h.x; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int p1, const float (&f)[2], R d, R dmin) {
        return mul_add(-dmin, (R)f[0], d * (R)((p0 << 3) + p1));
    }
};

template <> struct KR<T_Q5_K> {
    static constexpr int BYTES = BYTES_Q5_K, NCH = 11, NPL = 2, NF16 = 1;
    typedef u32x4 chunk_t;
    struct Hdr { u32x4 h, qh; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int hf) { return Hdr{row[0], row[1 + hf]}; }
    static constexpr int NEXT = 1;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int hf) { return Raw{row[3 + 4 * H + 2 * p + hf]}; }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int, u32x4 (&c)[2][2]) {
        uint32_t sc, mn;
        scale_min_pair(h.h, 2 * H + p, sc, mn);
        const uint32_t m0 = splat16(sc & 0xffu), m1 = splat16(sc >> 8), add = splat16(128u);
        const u32x4 q = r.q;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // bit 2*jp of qh[l] is the fifth bit of element 64*jp + l, bit 2*jp + 1 that of 64*jp + 32 + l
            // (reference ggml-quants.c:1460-1478); bits 5 to 7 are masked below
            const uint32_t t0 = H == 0 ? h.qh[i] << (4 - 2 * p) : h.qh[i] >> (2 * p), t1 = H == 0 ? h.qh[i] << (3 - 2 * p) : h.qh[i] >> (2 * p + 1);
            uint32_t hi, lo;
            byte_digits(merge_bits(0x0f0f0f0fu, q[i], t0), 0x001f001fu, m0, add, hi, lo);
            c[0][0][i] = hi; c[0][1][i] = lo;
            byte_digits(merge_bits(0x0f0f0f0fu, q[i] >> 4, t1), 0x001f001fu, m1, add, hi, lo);
            c[1][0][i] = hi; c[1][1][i] = lo;
        }
    }
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &h, int, int half) {
        uint32_t sc, mn;
        scale_min_quad(h.h, half, sc, mn);
        return bytes_to_f16_pairs(mn);
    }
    __device__ static __forceinline__ u32x2 f16_quad(const u32x4 *row, int g) {           // against the block sums 4g .. 4g + 3
        uint32_t sc, mn;
        scale_min_pair(row[0], g, sc, mn);
        return u32x2{f16_pair(mn & 0xffu, mn & 0xffu), f16_pair(mn >> 8, mn >> 8)};
    }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.h.x; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int p1, const float (&f)[2], R d, R dmin) {
        return mul_add(-dmin, (R)f[0], d * (R)((p0 << 8) + p1));
    }
};

template <> struct KR<T_Q6_K> {
    static constexpr int BYTES = BYTES_Q6_K, NCH = 14, NPL = 2, NF16 = 0;
    typedef u32x4_a2 chunk_t;
    // ql[128] | qh[64] | scales[16] | d: cells 0..7, 8..11, 12, and d in the last two bytes of cell 13.
    // Half h of a super-block holds, for l = 0..31, the elements 128h + 32b + l of k-blocks b = 0..3 as low / high nibble of
    // ql[64h + l] (b = 0 / 2) and of ql[64h + 32 + l] (b = 1 / 3), two more bits from qh[32h + l] >> 2b, scale
    // scales[8h + 2b + l/16]  (reference ggml-quants.c:1695-1711).  Item (h, p): k-blocks p and p + 2 of half h.
    struct Hdr { u32x4 sc; uint32_t d; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int) { return Hdr{row[12], row[13].w >> 16}; }
    static constexpr int NEXT = 2;
    struct Raw { u32x4 ql, qh; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int hf) {
        return Raw{row[4 * H + 2 * p + hf], row[8 + 2 * H + hf]};
    }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int hf, u32x4 (&c)[2][2]) {
        // scales[8h + 2p + hf] and scales[8h + 2p + 4 + hf]: byte 2p + hf of dwords 2h and 2h + 1
        const int s0 = (int8_t)(h.sc[2 * H] >> (16 * p + 8 * hf)), s1 = (int8_t)(h.sc[2 * H + 1] >> (16 * p + 8 * hf));
        const uint32_t sa = splat16((uint32_t)s0), ba = splat16((uint32_t)(128 - 32 * s0));
        const uint32_t sb = splat16((uint32_t)s1), bb = splat16((uint32_t)(128 - 32 * s1));
        const u32x4 ql = r.ql, qh = r.qh;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t t0 = qh[i] << (4 - 2 * p), t1 = qh[i] >> (2 * p);               // bits 4, 5 of every byte: the upper two bits
            const uint32_t q0 = merge_bits(0x0f0f0f0fu, ql[i], t0);                        // bits 6, 7 are masked below
            const uint32_t q1 = merge_bits(0x0f0f0f0fu, ql[i] >> 4, t1);
            uint32_t hi, lo;
            byte_digits(q0, 0x003f003fu, sa, ba, hi, lo);
            c[0][0][i] = hi; c[0][1][i] = lo;
            byte_digits(q1, 0x003f003fu, sb, bb, hi, lo);
            c[1][0][i] = hi; c[1][1][i] = lo;
        }
    }
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &, int, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.d; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int p1, const float (&)[2], R d, R) { return d * (R)((p0 << 8) + p1); }
};

template <> struct KR<T_Q3_K> {
    static constexpr int BYTES = BYTES_Q3_K, NCH = 7, NPL = 1, NF16 = 0;
    typedef u32x4_a2 chunk_t;
    // hmask[32] | qs[64] | scales[12] | d: cells 0, 1 and 2..5; cell 6 is bytes 94..109 (scales from its third byte, d at its end).
    // Element 128h + 32v + l: bits 2v of qs[32h + l], bit 4h + v of hmask[l], scale 8h + 2v + l/16.  Item (h, p): v = p and p + 2.
    struct Hdr { u32x4 hm; uint32_t s[3], d; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int hf) {
        const u32x4 t = row[6];
        Hdr h;
        h.hm = row[hf];
        h.s[0] = shr16(t.y, t.x); h.s[1] = shr16(t.z, t.y); h.s[2] = shr16(t.w, t.z);
        h.d = t.w >> 16;
        return h;
    }
    static constexpr int NEXT = 2;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int hf) { return Raw{row[2 + 2 * H + hf]}; }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int hf, u32x4 (&c)[2][1]) {
        // 6-bit scale 4w + i is byte i of word w (reference ggml-quants.c:1062-1071): words 2h and 2h + 1 hold k-blocks 0, 1 and 2, 3
        const uint32_t hi2 = h.s[2] >> (4 * H);
        const uint32_t wa = ((h.s[0] >> (4 * H)) & 0x0f0f0f0fu) | ((hi2 & 0x03030303u) << 4);
        const uint32_t wb = ((h.s[1] >> (4 * H)) & 0x0f0f0f0fu) | (((hi2 >> 2) & 0x03030303u) << 4);
        const int b = 16 * p + 8 * hf;
        const int sc[2] = {(int)((wa >> b) & 0xffu) - 32, (int)((wb >> b) & 0xffu) - 32};
        const u32x4 q = r.q;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int v = p + 2 * e;
            // byte = 128 + (4 - q)*sc in 0..252: the two bytes of a 16-bit lane never carry into each other, whatever the sign of
            // the multiplier (arithmetic modulo 2^16); flipping bit 7 gives the signed byte
            const uint32_t mul = splat16((uint32_t)(-sc[e])), add = splat16((uint32_t)((128 + 4 * sc[e]) * 0x101));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t hb = 4 * H + v < 2 ? h.hm[i] << (2 - 4 * H - v) : h.hm[i] >> (4 * H + v - 2);
                const uint32_t w = merge_bits(0x03030303u, q[i] >> (2 * v), hb) & 0x07070707u;
                c[e][0][i] = pk_mad16(w, mul, add) ^ 0x80808080u;
            }
        }
    }
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &, int, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.d; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int, const float (&)[2], R d, R) { return d * (R)-p0; }
};

template <> struct KR<T_Q2_K> {
    static constexpr int BYTES = BYTES_Q2_K, NCH = 6, NPL = 1, NF16 = 1;      // fp16 product: sum_j m_j * bsum_j over the 16 sub-blocks
    typedef u32x4_a4 chunk_t;
    // scales[16] (low nibble scale, high nibble min) | qs[64] | d | dmin: cells 0, 1..4, and d | dmin in the last dword of cell 5
    struct Hdr { u32x4 sc; uint32_t dd; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int) { return Hdr{row[0], row[5].w}; }
    static constexpr int NEXT = 2;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int hf) { return Raw{row[1 + 2 * H + hf]}; }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int hf, u32x4 (&c)[2][1]) {
        const int b = 16 * p + 8 * hf;
        const uint32_t s0 = (h.sc[2 * H] >> b) & 15u, s1 = (h.sc[2 * H + 1] >> b) & 15u;
        const u32x4 q = r.q;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            c[0][0][i] = ((q[i] >> (2 * p)) & 0x03030303u) * s0;                          // byte products <= 45
            c[1][0][i] = ((q[i] >> (2 * p + 4)) & 0x03030303u) * s1;
        }
    }
    // mins of sub-blocks 8 half .. 8 half + 7
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &h, int, int half) {
        const uint32_t a = half ? h.sc[2] : h.sc[0], b = half ? h.sc[3] : h.sc[1];
        u32x4 c;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = ((i < 2 ? a : b) >> (16 * (i & 1) + 4)) & 0x0f0fu;
            c[i] = f16_pair(w & 0xffu, w >> 8);
        }
        return c;
    }
    __device__ static __forceinline__ u32x2 f16_quad(const u32x4 *row, int g) {
        const uint32_t w = (reinterpret_cast<const uint32_t *>(row)[g] >> 4) & 0x0f0f0f0fu;
        return u32x2{f16_pair(w & 0xffu, (w >> 8) & 0xffu), f16_pair((w >> 16) & 0xffu, w >> 24)};
    }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.dd; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int, const float (&f)[2], R d, R dmin) {
        return mul_add(-dmin, (R)f[0], d * (R)p0);
    }
};

template <> struct KR<T_IQ4_XS> {
    static constexpr int BYTES = BYTES_IQ4_XS, NCH = 9, NPL = 2, NF16 = 0;
    typedef u32x4_a4 chunk_t;
    // d | u16 scales_h | scales_l[4] | qs[128]: sub-block ib is qs[16 ib ..], low nibbles elements 0..15, high nibbles 16..31.
    // Cells 0..7 are bytes 0..127, cell 8 bytes 120..135 (sub-block 7).  Item (H, p): sub-blocks 4H + 2p and the next.
    struct Hdr { u32x2 h; };
    __device__ static __forceinline__ Hdr hdr(const u32x4 *row, int) { return Hdr{*reinterpret_cast<const u32x2 *>(row)}; }
    static constexpr int NEXT = 1;
    struct Raw { u32x2 q[4]; };
    __device__ static __forceinline__ Raw load(const u32x4 *row, int H, int p, int) {
        Raw r;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int ib = 4 * H + 2 * p + e;
            const u32x2 *qp = reinterpret_cast<const u32x2 *>(row) + (ib < 7 ? 1 + 2 * ib : 16);
            r.q[2 * e] = qp[0];
            r.q[2 * e + 1] = qp[1];
        }
        return r;
    }
    __device__ static __forceinline__ void expand(const Raw &r, const Hdr &h, int H, int p, int hf, u32x4 (&c)[2][2]) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int ib = 4 * H + 2 * p + e;
            const int ls = iq4_xs_scale(h.h, ib);
            const uint32_t mul = splat16((uint32_t)ls), add = splat16((uint32_t)(128 - 128 * ls));
            const uint32_t w[4] = {r.q[2 * e].x, r.q[2 * e].y, r.q[2 * e + 1].x, r.q[2 * e + 1].y};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t hi, lo;
                byte_digits(iq4_codes((w[i] >> (4 * hf)) & 0x0f0f0f0fu), 0x00ff00ffu, mul, add, hi, lo);
                c[e][0][i] = hi; c[e][1][i] = lo;
            }
        }
    }
    __device__ static __forceinline__ u32x4 f16_cell(const Hdr &, int, int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ static __forceinline__ uint32_t scales(const Hdr &h) { return h.h.x & 0xffffu; }
    template <typename R> __device__ static __forceinline__ R value(int p0, int p1, const float (&)[2], R d, R) { return d * (R)((p0 << 8) + p1); }
};

// k-block e (0, 1) of item (H, p)
template <class T> __device__ __forceinline__ constexpr int kr_k_block(int H, int p, int e) { return 4 * H + (3 - T::NEXT) * p + T::NEXT * e; }

}  // namespace
}  // namespace chip
