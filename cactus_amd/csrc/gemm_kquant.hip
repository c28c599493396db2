// Prefill GEMM for gfx950 over K-quant weights (Q2_K .. Q6_K, IQ4_XS) and Q8_K activations: the batched form of
// lm_ggml_vec_dot_q2_K_q8_K .. _q6_K_q8_K, _iq4_xs_q8_K (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// This file holds the choice of the kernel and the staging kernel, which runs Q6_K, Q3_K and IQ4_XS where there is a tile for at most every CU;
// gemm_kr_kernel (gemm_kquant_rows.hip) runs everything else.
//
// Per 256-value super-block the reference forms sumi = sum_j sc_j * dot(q_j, a_j) with signed scales per 16 values, and applies d
// and the activation scale once.  The integer scales are folded into the int8 MFMA operand: Q6_K as the two signed bytes of (q - 32)*sc =
// 256*hi + lo, sumi = 256*P0 + P1, as those of code*sc of IQ4_XS; Q3_K as one plane (4 - q)*sc in -128..124, sumi = -P0.  The planes accumulate in the MFMA's own int32
// accumulator over the 8 k-blocks of a super-block, all sums are exact, and the vector unit works once per super-block and output.
//
// Measured for Q6_K with these digits against base-64 digits of the product plus 4064 (16 instead of 10 vector instructions per four weights, and a
// correction by the block sums), us: 14336 values x 4096 rows at 512 tokens 129 -> 113, 4096 x 4096 at 512 tokens 43 -> 38.6.
//
// Structure: a workgroup of WR x WC waves owns 32*WR rows x 64*WC tokens; each wave owns one 32-row tile by two
// 32-token tiles.  LDS is double buffered over stages of 4 k-blocks (half a super-block), one barrier per stage.
// Operand cells are 16 bytes ([plane][k-block][k-half][row]), exactly what one lane feeds v_mfma_i32_32x32x32_i8.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include "kquant_dev.h"
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace chip {

constexpr int KQ_KB = 4;                      // 32-value k-blocks per LDS stage
constexpr int KQ_TN = 2;                      // 32-token tiles per wave

// One staging item = (row, x) of a stage h (half of a super-block): p = x / 2, the 16 values hf = x & 1 of k-blocks p and p + 2 of that
// half, which expand into one operand cell per digit plane and k-block.
template <int WT> struct KQ;

template <> struct KQ<T_Q6_K> {
    static constexpr int BYTES = BYTES_Q6_K, NPL = 2;              // int8 digit planes
    // Half h of a super-block holds, for l = 0..31, the elements 128h + 32b + l of k-blocks b = 0..3 as
    //   low / high nibble of ql[64h + l] (b = 0 / 2) and of ql[64h + 32 + l] (b = 1 / 3), two more bits from
    //   qh[32h + l] >> 2b, scale scales[8h + 2b + l/16]                       (reference ggml-quants.c:1695-1711)
    struct Raw { u32x4 ql[2], qh[2], sc; uint32_t d; };
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
    __device__ static __forceinline__ void expand(u32x4 (&cell)[NPL][2], const Raw &r, int h, int x) {
        const int p = x >> 1, hf = x & 1;
        // scales[8h + 2p + hf] and scales[8h + 2p + 4 + hf]: byte 2p + hf of dwords 2h and 2h + 1
        const int s0 = __builtin_amdgcn_sbfe((int)r.sc[2 * h], 8 * (2 * p + hf), 8);
        const int s1 = __builtin_amdgcn_sbfe((int)r.sc[2 * h + 1], 8 * (2 * p + hf), 8);
        const uint32_t sa = splat16((uint32_t)s0), ba = splat16((uint32_t)(128 - 32 * s0));
        const uint32_t sb = splat16((uint32_t)s1), bb = splat16((uint32_t)(128 - 32 * s1));
        const u32x4 ql = r.ql[h], qh = r.qh[h];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t hb = qh[i] >> (2 * p);                                               // bits 0, 1 / 4, 5: the upper two bits
            uint32_t hi, lo;
            byte_digits(merge_bits(0x0f0f0f0fu, ql[i], hb << 4), 0x003f003fu, sa, ba, hi, lo);  // k-block p
            cell[0][0][i] = hi; cell[1][0][i] = lo;
            byte_digits(merge_bits(0x0f0f0f0fu, ql[i] >> 4, hb), 0x003f003fu, sb, bb, hi, lo);  // k-block p + 2
            cell[0][1][i] = hi; cell[1][1][i] = lo;
        }
    }
    __device__ static __forceinline__ int sumi(int p0, int p1) { return (p0 << 8) + p1; }
};

template <> struct KQ<T_Q3_K> {
    static constexpr int BYTES = BYTES_Q3_K, NPL = 1;
    // hmask[32] | qs[64] | scales[12] | d.  Element 128h + 32v + l: bits 2v of qs[32h + l], bit 4h + v of hmask[l], scale 8h + 2v + l/16.
    // The two items of a k-half read the same bytes.
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
    __device__ static __forceinline__ void expand(u32x4 (&cell)[NPL][2], const Raw &r, int h, int x) {
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
                const uint32_t q = merge_bits(0x03030303u, r.q[h][i] >> (2 * v), (r.hm[i] >> (4 * h + v)) << 2) & 0x07070707u;
                cell[0][c][i] = pk_mad16(q, mul, add) ^ 0x80808080u;
            }
        }
    }
    __device__ static __forceinline__ int sumi(int p0, int) { return -p0; }
};

template <> struct KQ<T_IQ4_XS> {
    static constexpr int BYTES = BYTES_IQ4_XS, NPL = 2;
    // d | u16 scales_h | scales_l[4] | qs[128]: k-block ib is qs[16 ib ..], low nibbles its first k-half, high nibbles the second.
    // The two items of a k-block read the same bytes.
    struct Raw { u32x4 q[2][2]; u32x2 h; uint32_t d; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *blk, int x) {
        const int p = x >> 1;
        r.h = *reinterpret_cast<const u32x2 *>(blk);
        r.d = r.h.x & 0xffffu;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int c = 0; c < 2; c++) r.q[h][c] = *reinterpret_cast<const u32x4_a4 *>(blk + 8 + 16 * (4 * h + p + 2 * c));
    }
    __device__ static __forceinline__ void expand(u32x4 (&cell)[NPL][2], const Raw &r, int h, int x) {
        const int p = x >> 1, hf = x & 1;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int ls = iq4_xs_scale(r.h, 4 * h + p + 2 * c);
            const uint32_t mul = splat16((uint32_t)ls), add = splat16((uint32_t)(128 - 128 * ls));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t hi, lo;
                byte_digits(iq4_codes((r.q[h][c][i] >> (4 * hf)) & 0x0f0f0f0fu), 0x00ff00ffu, mul, add, hi, lo);
                cell[0][c][i] = hi; cell[1][c][i] = lo;
            }
        }
    }
    __device__ static __forceinline__ int sumi(int p0, int p1) { return (p0 << 8) + p1; }
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
    static constexpr int NPL = T::NPL;
    // plane stride 2 mod 16 cells: the staging threads of one wave spread over the bank groups
    static constexpr int A_PLANE = BM + 2, B_PLANE = BN + 2;
    static constexpr int A_CELLS = NPL * KQ_KB * 2 * A_PLANE;   // 16-byte cells
    static constexpr int B_CELLS = KQ_KB * 2 * B_PLANE;
    // one stage buffer (two of them, by stage parity)
    static constexpr size_t OFF_A = 0;
    static constexpr size_t OFF_B = OFF_A + (size_t)A_CELLS * 16;
    static constexpr size_t STAGE = OFF_B + (size_t)B_CELLS * 16;
    // one super-block buffer (two of them, by super-block parity)
    static constexpr size_t OFF_SD = 0;                                     // u32 [BM]: d, permuted per 32 rows
    static constexpr size_t OFF_SX = OFF_SD + (size_t)BM * 4;               // f32 [BN]: activation scale of the super-block
    static constexpr size_t SBLK = OFF_SX + (size_t)BN * 4;
    static constexpr size_t OFF_STAGES = 0;
    static constexpr size_t OFF_SBLK = 2 * STAGE;
    static constexpr size_t OFF_DUMP = OFF_SBLK + 2 * SBLK;                 // 16 bytes per staging thread: where stores that do not apply go
    static constexpr size_t TOTAL = OFF_DUMP + (size_t)NPT * 16;
    static constexpr int W_ITEMS = BM * 4;
    static constexpr int W_PER_T = W_ITEMS / NPT;
    static constexpr int X_ITEMS = BN * KQ_KB * 2;
    static constexpr int X_PER_T = X_ITEMS / NPT;
    static_assert(BN <= NPT, "a staging thread per token fetches its scale");
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
    // split K: grid row s takes super-blocks sb0 .. of every row
    // and writes its partial tile to slice s of y
    int sb0 = 0, nstages = (int)(K / QK_K) * 2;
    if (!GATHER && slice_sb > 0) {
        sb0 = (int)blockIdx.y * slice_sb;
        nstages = 2 * min(slice_sb, (int)(K / QK_K) - sb0);
        y += (size_t)blockIdx.y * (size_t)M * (size_t)ldy;
    }
    TileCoord tc;
    int32_t entry = 0;
    if constexpr (GATHER) {
        if (!gather_tile<C::BN>(rg, map, entry, tc.row_tile)) return;
        tc.tok_tile = 0;
    } else {
        tc = xcd_tile(blockIdx.x, map);
        if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;    // padding of the tile map
    }
    size_t w_offset;
    const GatherView gv = resolve_gather<GATHER>(rg, entry, w_offset, M);
    W += w_offset;
    const int64_t row_base = (int64_t)tc.row_tile * C::BM;
    const int64_t tok_base = (int64_t)(GATHER ? gv.tok_tile : tc.tok_tile) * C::BN;
    if (tok_base >= M) return;

    if (wave >= C::NC) {
        // ------------------------------------------------------------------------------------ staging waves
        const int pt = tid - C::NC * 64;
        const size_t off_d = q8_K_off_d(K);
        uint8_t *const dump = lds + C::OFF_DUMP + pt * 16;
        struct Acts {
            u32x4 x[C::X_PER_T];
            float xs;
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
        // activation scale: thread t < BN for token t
        const uint8_t *ssrc = ws + (size_t)gv.act_row(min(tok_base + min(pt, C::BN - 1), M - 1)) * ws_stride;
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
                u32x4 cell[C::NPL][2];
                T::expand(cell, RW.w[i], h, x);
                const int c0 = (x >> 1) * 2 + (x & 1), c1 = c0 + 4;       // [k-block][k-half]
#pragma unroll
                for (int pl = 0; pl < C::NPL; pl++) {
                    A[(pl * KQ_KB * 2 + c0) * C::A_PLANE + r] = cell[pl][0];
                    A[(pl * KQ_KB * 2 + c1) * C::A_PLANE + r] = cell[pl][1];
                }
                if constexpr (even) {
                    // the lane that owns MFMA result register v of a 32-row tile holds row 8*(v/4) + 4*half + v%4:
                    // keep the scale of row i at half*16 + (i/8)*4 + i%4 so a lane reads its 16 scales contiguously
                    const int i32 = r & 31;
                    const int pos = ((i32 >> 2) & 1) * 16 + (i32 >> 3) * 4 + (i32 & 3);
                    uint8_t *dst = (x == 0) ? sblk + C::OFF_SD + ((r & ~31) + pos) * 4 : dump;
                    *reinterpret_cast<uint32_t *>(dst) = RW.w[i].d;
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

    // once per super-block: fold the planes, out += d * float(sumi) * dx
    auto fold = [&](int sbp) {
        const uint8_t *sblk = lds + C::OFF_SBLK + (size_t)sbp * C::SBLK;
        const u32x4 *sp = reinterpret_cast<const u32x4 *>(sblk + C::OFF_SD) + (r0 + half * 16) / 4;
        const u32x4 s0 = sp[0], s1 = sp[1], s2 = sp[2], s3 = sp[3];
        const uint32_t sd[16] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w, s2.x, s2.y, s2.z, s2.w, s3.x, s3.y, s3.z, s3.w};
#pragma unroll
        for (int c = 0; c < TN; c++) {
            const float dx = reinterpret_cast<const float *>(sblk + C::OFF_SX)[n0 + c * 32 + l32];
#pragma unroll
            for (int v = 0; v < 16; v++) out[c][v] = __builtin_fmaf(h2f(sd[v]) * (float)T::sumi(P[0][c][v], P[C::NPL - 1][c][v]), dx, out[c][v]);
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
// Slices of K over the grid's second dimension, each a serial walk whose partial outputs are added in order: for 64 rows x 128 tokens up to
// two workgroups per CU with one token tile, one per CU with more (the partial outputs grow with the token count), at least four
// super-blocks each.  The same for both kernels, so that the bits of a product do not depend on which one runs it.
static int kq_slices_for(int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int64_t units = K / QK_K, tiles = ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)128);
    if (units < 8 || (M <= 128 && !kq_splittable(N))) return 1;
    const int64_t s = std::min({(M <= 128 ? 2 : 1) * cus / tiles, units / 4, (int64_t)16});
    if (s < 2) return 1;
    const int64_t per = ceil_div(units, s);
    return (int)ceil_div(units, per);                                   // no empty slice
}
// How a product is covered: the staging kernel (groups 0), or gemm_kr_kernel in one or two k groups a workgroup (1: four waves that walk the
// super-blocks in order, two workgroups a CU; 2: eight waves, four on the even and four on the odd super-blocks, one workgroup a CU); and slices of K.
// Q3_K .. Q6_K run in the slices above, mostly in one group - or, Q6_K and Q3_K with at most a 128 x 64 tile for every CU, in the staging kernel,
// which expands a weight once for 128 tokens (us, staged / gemm_kr_kernel: Q6_K 14336 values x 4096 rows at 512 tokens 113 / 128, 201 tokens 66 / 74,
// 4096 x 4096 at 512 tokens 38.6 / 44; Q3_K 14336 x 4096 at 201 tokens 49 / 53), unless half of its 128-token tile would be empty and the slices
// give gemm_kr_kernel a workgroup for every CU (32 tokens: Q6_K 41 / 27, Q3_K 30 / 20).
// Rows above 2048 values whose workgroups fit the CUs take two groups a workgroup where one would leave a CU four waves (us, one / two groups: Q4_K unsplit
// 4096 x 4096 at 512 tokens 32.8 / 28.3, 14336 rows at 64 27.8 / 25.0; Q5_K 36.9 / 32.3; over 700 products 1.12 x, none slower; up to 2048 values 1.01
// x and one group stays) or where the staging kernel's tiles come to a second turn (Q6_K 1.57 x, Q3_K 1.84 x over 44 products: 128-token tiles
// that are half empty); Q3_K above 128 tokens on half the CUs and more in any case (14336 x 4096 at 201 tokens 42.3 / 40.3 without the quantizer; 1.05 x).
// Q2_K and IQ4_XS by their number of 128 x 64 tiles:
//   more tiles than CUs     one group (us, 512 tokens x 4096 values x 4608 rows, one / two groups: Q2_K 36 / 44, IQ4_XS 66 / 72)
//   above half as many      two groups, so that every SIMD has two waves (4096 rows: Q2_K 29 / 27, IQ4_XS 45 / 42); so too with 2 slices of
//                           rows above 8192 values (14336 values x 4096 rows at 201 tokens: Q2_K 47 / 42, IQ4_XS 75 / 68)
//   fewer                   as many slices as give every CU a workgroup, at most 8, or 16 of four super-blocks (a slice more costs its
//                           partial outputs: Q2_K 14336 values x 4096 rows at 64 tokens 68, 42, 29, 23, 26 us in 1, 2, 4, 8, 12).  Not
//                           rounded up: 96 tiles in 3 slices leave 32 workgroups for a second turn (IQ4_XS 4096 x 4096 at 130 tokens 29 / 31 us
//                           in 2 / 3).  The slice sum pays for at most 150000 partial outputs a super-block of a row (IQ4_XS 1792 values x
//                           4096 rows at 64 tokens 21.7 / 16.4 whole / in 4), not for rows of three or less or for two slices of less than 8.
//   IQ4_XS, 5 to 11 super-blocks in one or two slices, up to 128 tokens: the staging kernel (us, staged / gemm_kr_kernel: 2304 values x
//                           8192 rows at 93 tokens 21.5 / 25.9, 1280 x 8192 at 64 16.3 / 19.0; 2560 x 15500 at 127 31.3 / 29.4); 2 and 3 up
//                           to 96 tokens on at most 1000000 outputs, 600000 where the other kernel has one token tile (768 x 3788 at 52 11.7 / 12.8,
//                           512 x 11088 at 65 10.7 / 11.9; 512 x 14373 at 60 12.2 / 11.5, 512 x 13107 at 86 13.5 / 12.2)
struct KqPlan { int groups, slices; };
static KqPlan kq_plan(int wtype, int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int64_t tiles = ceil_div(N, (int64_t)128) * ceil_div(M, (int64_t)64), units = K / QK_K;
    if (wtype != T_Q2_K && wtype != T_IQ4_XS) {
        const int slices = kq_slices_for(K, N, M, cus);
        const bool staged = (wtype == T_Q6_K || wtype == T_Q3_K) && tiles <= cus && (M > 64 || tiles * slices < cus);
        const bool fits = units > 8 && tiles * slices <= cus;
        const bool two = fits && (wtype == T_Q4_K || wtype == T_Q5_K ? slices == 1
                                                                     : staged && (ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)128) * slices > cus ||
                                                                                  (wtype == T_Q3_K && M > 128 && 2 * tiles * slices >= cus)));
        return KqPlan{two ? 2 : staged ? 0 : 1, slices};
    }
    if (tiles > cus || units == 1) return KqPlan{1, 1};
    const int64_t most = std::max<int64_t>(8, std::min<int64_t>(16, units / 4));
    int64_t s = units < 4 ? 1 : std::min({cus / tiles, units, most, units * 150000 / (M * N)});
    if (s < (units < 8 ? 3 : 2)) s = 1;
    if (wtype == T_IQ4_XS && units < 4 && M <= 96 && M * N <= (M > 64 ? 1000000 : 600000)) return KqPlan{0, 1};
    if (wtype == T_IQ4_XS && s <= 2 && units >= 5 && units < 12 && M > (units < 8 ? 32 : 64) && M <= 128 && M * N <= 1400000) return KqPlan{0, kq_slices_for(K, N, M, cus)};
    if (s == 1) return KqPlan{units < 4 ? 1 : 2, 1};
    const int64_t per = ceil_div(units, s);
    s = ceil_div(units, per);                                           // no empty slice
    return KqPlan{s == 2 && units > 32 ? 2 : 1, (int)s};
}

// With few tokens the GEMM's time is its walk over K, whatever the token count, while the GEMV forms pass over the weights once
// per 8 (Q6_K) or 16 tokens (Q4_K, Q5_K) at memory speed.  With K in slices, or on rows too short for them, the GEMM is ahead from the first
// token of a second pass on (us, GEMV passes / GEMM: Q4_K at 17 tokens 4096 x 4096 17.4 / 15.1, at 33 tokens 1536 values x 2048 rows 31 / 15,
// at 18 tokens 512 x 4096 12 / 9.5; Q6_K at 17 tokens 1280 x 8192 34 / 16).  On matrices with too many rows to split Q4_K and Q5_K stay with a
// second pass (14336 rows x 4096 values at 24 tokens 27.7 / 27.5), and where the caller's workspace has no room for the partial outputs
// the unsplit walk pays later.
static int64_t gemm_kq_min_tokens(int wtype, int64_t K, int64_t N, bool can_split) {
    const bool q6 = wtype == T_Q6_K, long_rows = K > 8192;
    if (can_split) return q6 ? 9 : 17;
    if (!kq_splittable(N)) return q6 ? 9 : 33;
    if (K < 8 * QK_K) return q6 ? 9 : 17;
    return q6 ? (long_rows ? 41 : 25) : (long_rows ? 33 : 49);
}

// Q3_K, Q2_K and IQ4_XS: the dot-product GEMV passes of 8 tokens, whose time grows with the tokens, against the GEMM, whose time
// below 128 tokens does not.  A token count alone does not part them (GEMV / GEMM, us, rows x values, split K: Q3_K 300 x 2816
// at 10 tokens 11 / 14, 4096 x 4096 at 9 tokens 15 / 14, 1024 x 14336 at 9 tokens 19 / 14; IQ4_XS 1024 x 4096 at 10 tokens 12 / 13, 8192 x 8192 at 12
// tokens 37 / 27; unsplit: IQ4_XS 748 x 7168 at 32 tokens 33 / 48, 4096 x 1024 at 25 tokens 31 / 13), so both times are estimated, in us.
// The terms of the GEMM were fitted to the staging kernel in the slices of kq_slices_for, which Q2_K and IQ4_XS only rarely run in now: for them
// they are an upper bound, and the GEMM is taken late rather than early.  Of 5100 products (9 to 200 tokens, values x rows, GEMV / GEMM)
// the slower one is taken by more than 5 per cent in 1 per cent of Q3_K (2048 x 290 at 10 tokens 11.3 / 14.2), 4 of Q2_K (8192 x 9071 at 14 tokens
// 46 / 22) and 6 of IQ4_XS (9984 x 10019 at 14 tokens 60 / 34), nearly always the GEMV:
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
        return low_bit_gemm_ahead(wtype, K, N, n, can_split ? kq_slices_for(K, N, n, 256) : 1);
    return n >= gemm_kq_min_tokens(wtype, K, N, can_split);
}
int gemm_kq_slices(int wtype, int64_t K, int64_t N, int64_t n, int compute_units) {
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    if (!gemm_kq_supported(wtype, K, N, n, true)) return 1;
    return kq_plan(wtype, K, N, n, cus).slices;
}

// gemm_kq_few_kernel against whatever else would run the product: both times are estimated, in us, and it is taken where it is ahead by 7 per cent.
// Fitted to 12500 products (512 to 14336 values, 256 to 20000 rows, 5 to 300 tokens; each with up to five forms of this kernel), which it is within 7 per
// cent of (the others within 5 to 10; the matrix-core GEMVs 23).  Over the same products: 5 to 8 tokens 1.28 x, 9 to 16 1.78, 17 to 32 1.56, 33 to
// 64 1.42, to 128 1.32, to 300 1.20; the best form that there is would be 1 to 2 per cent faster still; one product in 110 is more than 3 per cent slower.
//   fixed, turn   launch, first loads and the sum of the waves; once more per turn of the workgroups that fit the device
//   walk          a super-block of one wave after the other
//   work, cu      vector instructions: super-blocks per SIMD, on average and on the busiest CU
struct FewForm { int rt, tt, ks; float fixed, turn, walk, work, cu; };
static constexpr FewForm kFewForms[] = {
    {1, 1, 4, 2.764f, 0.553f, 0.249f, 0.235f, 0.377f}, {1, 1, 8, 2.582f, 0.780f, 0.071f, 0.159f, 0.483f}, {1, 1, 16, 1.795f, 1.679f, 0.111f, 0.173f, 0.473f},
    {2, 1, 2, 0.f, 3.677f, 0.607f, 0.370f, 0.780f},    {2, 1, 4, 0.f, 3.803f, 0.390f, 0.415f, 0.643f},    {1, 2, 4, 3.117f, 1.037f, 0.252f, 0.169f, 0.517f},
    {1, 2, 8, 2.062f, 1.785f, 0.090f, 0.156f, 0.640f}, {2, 2, 2, 4.216f, 0.818f, 0.843f, 0.206f, 0.788f}, {2, 2, 4, 4.119f, 0.896f, 0.487f, 0.274f, 0.798f},
    {2, 2, 8, 2.349f, 1.802f, 0.438f, 0.211f, 1.005f}};
// a type's share of the walk and the work; the GEMMs: fixed, slices of K, a walk's super-block, a turn, super-blocks per workgroup slot, the walk of a
// second token tile, a million partial outputs; the dot-product GEMV: a pass, its rounds of 1024 rows, then per token parts of 4096 values, those times the
// rounds, and the same per pass; the matrix-core GEMV: a pass, its steps of 16 rows a CU, 1e4 values per pass, 1e5 per token, steps per 10 tokens
struct KqTimes { float few, gemm[7], gemv[5], mmv[5]; };
static const KqTimes &kq_times(int wtype) {
    static const KqTimes q4k{0.936f, {2.946f, 2.733f, 0.783f, 2.216f, 1.611f, 0.353f, 1.469f}, {3.178f, 0.f, 0.108f, 0.132f, 0.f}, {5.602f, 0.f, 0.f, 2.018f, 0.785f}};
    static const KqTimes q5k{1.206f, {1.790f, 2.643f, 1.163f, 3.531f, 1.524f, 0.357f, 1.793f}, {3.051f, 0.f, 0.120f, 0.118f, 0.211f}, {5.714f, 0.093f, 0.f, 2.391f, 0.836f}};
    static const KqTimes q6k{1.284f, {2.948f, 2.387f, 1.055f, 2.261f, 1.456f, 0.231f, 2.027f}, {3.437f, 0.207f, 0.126f, 0.105f, 0.075f}, {}};
    static const KqTimes q3k{0.887f, {2.393f, 2.177f, 0.744f, 2.435f, 1.179f, 0.251f, 1.955f}, {3.182f, 0.271f, 0.135f, 0.093f, 0.120f}, {}};
    static const KqTimes q2k{0.85f, {4.631f, 2.364f, 0.616f, 0.f, 1.671f, 0.321f, 1.015f}, {3.041f, 0.218f, 0.140f, 0.114f, 0.f}, {}};
    static const KqTimes iq4{1.348f, {5.142f, 2.518f, 1.090f, 0.f, 2.777f, 0.418f, 0.816f}, {2.961f, 0.232f, 0.146f, 0.107f, 0.017f}, {}};
    switch (wtype) {
        case T_Q4_K: return q4k;
        case T_Q5_K: return q5k;
        case T_Q6_K: return q6k;
        case T_Q3_K: return q3k;
        case T_Q2_K: return q2k;
        default:     return iq4;
    }
}
static float few_estimate(const FewForm &f, int wtype, int64_t K, int64_t N, int64_t n, int64_t cus) {
    const int64_t units = K / QK_K, blocks = ceil_div(N, (int64_t)(16 * f.rt)) * ceil_div(n, (int64_t)(16 * f.tt));
    const int simd = f.rt * f.tt == 1 ? 4 : f.rt * f.tt == 2 ? 3 : 2;                    // waves a SIMD's registers hold
    const int64_t slots = cus * std::max<int64_t>(1, std::min(160 * 1024 / (gemm_kq_few_stretch(wtype, f.rt, f.tt) * f.ks), 4 * simd / f.ks));
    const float turns = (float)ceil_div(blocks, slots);
    return f.fixed + f.turn * turns + kq_times(wtype).few * (f.walk * turns * (float)ceil_div(units, (int64_t)f.ks) + f.work * (float)(blocks * units) / (float)(4 * cus) +
                                                             f.cu * (float)(ceil_div(blocks, cus) * units) / 4.f);
}
// the GEMM, the matrix-core GEMV (Q4_K, Q5_K) or the dot-product GEMV, whichever a caller with room for partial outputs would reach
static float others_estimate(int wtype, int64_t K, int64_t N, int64_t n, const KqPlan &p, int64_t cus) {
    const KqTimes &t = kq_times(wtype);
    const bool four = wtype == T_Q4_K || wtype == T_Q5_K;
    const int64_t units = K / QK_K;
    if (four ? n >= gemm_kq_min_tokens(wtype, K, N, p.slices > 1) : n >= 9) {
        const int64_t tiles = p.groups == 0 ? ceil_div(N, (int64_t)64) * ceil_div(n, (int64_t)128) : ceil_div(N, (int64_t)128) * ceil_div(n, (int64_t)64);
        const int64_t per = ceil_div(ceil_div(units, (int64_t)p.slices), (int64_t)(p.groups == 2 ? 2 : 1));
        const float turns = (float)ceil_div(tiles * p.slices, cus * (p.groups == 1 ? 2 : 1)), walk = turns * (float)per;
        return t.gemm[0] + (p.slices > 1 ? t.gemm[1] + t.gemm[6] * (float)p.slices * (float)(N * n) * 1e-6f : 0.f) + (t.gemm[2] + (n > 32 ? t.gemm[5] : 0.f)) * walk +
               t.gemm[3] * turns + t.gemm[4] * (float)(tiles * units) / (float)(2 * cus);
    }
    if (four && n >= (N * K >= (32LL << 20) ? 5 : 7)) {
        const float passes = (float)ceil_div(n, (int64_t)(K <= 6144 ? 16 : 8)), steps = (float)ceil_div(ceil_div(ceil_div(N, (int64_t)16), cus) * units, (int64_t)8);
        return passes * (t.mmv[0] + t.mmv[1] * steps + t.mmv[2] * 1e-4f * (float)K) + (float)n * (t.mmv[3] * 1e-5f * (float)K + t.mmv[4] * 0.1f * steps);
    }
    const float passes = (float)ceil_div(n, (int64_t)8), rounds = (float)ceil_div(N, (int64_t)1024), parts = (float)ceil_div(K, (int64_t)4096);
    return passes * (t.gemv[0] + t.gemv[1] * rounds + t.gemv[4] * parts * rounds) + (float)n * parts * (t.gemv[2] + t.gemv[3] * rounds);
}
// Forms of 32 tokens above 16 tokens.  Rows of two super-blocks up to 32 tokens, of three there for the types without a matrix-core GEMV, from four on
// otherwise: K is what the waves share.  Above 32 tokens a caller without room for slices of K keeps the order of one walk over it.  Products that
// are known to run in slices of K and a slice sum stay there: long rows on many rows (us, slices / this, 14336 values x 4096 rows at 32 tokens: Q4_K 19.8
// / 18.9, Q6_K 23.9 / 20.8, Q3_K 19.6 / 16.8) and a few rows above 64 tokens.  So do Q6_K and Q3_K above 32 tokens whose tiles in the staging kernel come to
// two thirds and three quarters of the CUs, where 39 products are 0.96 x its speed (Q6_K 1024 values x 11884 rows at 49 tokens 11.6 / 13.4, 3328 x 16161
// at 47 26.8 / 29.2; Q3_K 1536 x 13500 at 33 11.4 / 13.5; just below 38 are 1.07 x).  Up to 1200 tokens: beyond the 300 of the fit the estimates
// are extrapolated (1464 products of 300 to 1200 tokens 1.17 x).
KqFew kq_few_plan(int wtype, size_t nb01, int64_t K, int64_t N, int64_t n, bool can_split, int compute_units) {
    if (!gemm_kq_type(wtype) || n < 5 || n > 1200 || N < 1 || K % QK_K != 0) return KqFew{0, 0, 0};
    // rows that the kernel's 32-bit offsets reach from a tile's first: forms of 32 rows where all of them are, none where not even 16 are
    const int64_t reach = gemm_kr_rows_in_reach(nb01);
    if (reach < 16) return KqFew{0, 0, 0};
    const int64_t cus = compute_units > 0 ? compute_units : 256, units = K / QK_K, forced = tune("CHIP_KQ_FEW", -1);
    if (forced > 0) return units >= forced % 100 && reach >= 16 * (forced / 1000) ? KqFew{(int)(forced / 1000), (int)(forced / 100 % 10), (int)(forced % 100)} : KqFew{0, 0, 0};
    const bool four = wtype == T_Q4_K || wtype == T_Q5_K;
    if (forced == 0 || units < (n <= 32 ? 2 : 4) || (units == 3 && four) || tune("CHIP_GEMM_MIN_TOKENS", 0) > 0) return KqFew{0, 0, 0};
    const KqPlan p = kq_plan(wtype, K, N, n, cus);
    if (n > 32 && p.slices > 1 && !can_split) return KqFew{0, 0, 0};
    if (p.slices > 1 && ((n > 16 && K > 8192 && N > 2048) || (n > 64 && N < 320))) return KqFew{0, 0, 0};
    if (const int64_t staged = ceil_div(N, (int64_t)64) * ceil_div(n, (int64_t)128); p.groups == 0 && p.slices == 1 && n > 32 &&
        (wtype == T_Q6_K ? 3 * staged >= 2 * cus : wtype == T_Q3_K && 4 * staged >= 3 * cus)) return KqFew{0, 0, 0};
    KqFew best{0, 0, 0};
    float least = 0.93f * others_estimate(wtype, K, N, n, p, cus);
    for (const FewForm &f : kFewForms) {
        // (at most eight super-blocks a wave: a chain of eight additions at most, gemm_kquant_few.hip)
        if (f.tt != (n > 16 ? 2 : 1) || f.ks > units || units > 8 * f.ks || reach < 16 * f.rt) continue;
        if (const float e = few_estimate(f, wtype, K, N, n, cus); e < least) { least = e; best = KqFew{f.rt, f.tt, f.ks}; }
    }
    return best;
}

using KqTile = KqCfg<T_Q6_K, 2, 2>;                                          // 64 x 128, 4 + 4 waves
template <int WT, bool GATHER>
static hipError_t launch_kq(const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride, int64_t M,
                            float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather &rg, int64_t slots, int slices, float *part) {
    using C = KqCfg<WT, 2, 2>;
    const size_t lds_bytes = C::TOTAL;
    if ((int64_t)lds_bytes > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kq_kernel<WT, 2, 2, 2, GATHER>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, lds_bytes, lim, grant); e != hipSuccess) return e;
    const TileMap map = make_tile_map(ceil_div(N, C::BM), GATHER ? 1 : ceil_div(M, C::BN), 32);     // 32 workgroups run on an XCD at a time
    const int slice_sb = slices > 1 ? (int)ceil_div(K / QK_K, (int64_t)slices) : 0;
    hipLaunchKernelGGL(kfn, GATHER ? gather_grid(map, slots, C::NT) : dim3(map.grid, (unsigned)slices), dim3(C::NT), lds_bytes, st, (const uint8_t *)W,
                       nb01, K, N, (const uint8_t *)ws, ws_stride, M, slices > 1 ? part : y, slices > 1 ? N : ldy, map, rg, slice_sb);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return slices > 1 ? launch_sum_slices(part, slices, M, N, y, ldy, st) : hipSuccess;
}

template <bool GATHER>
static hipError_t launch_staged_type(int wtype, const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride, int64_t M, float *y,
                                     int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather &rg, int64_t slots, int slices, float *part) {
    switch (wtype) {
        case T_Q6_K: return launch_kq<T_Q6_K, GATHER>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, slots, slices, part);
        case T_Q3_K: return launch_kq<T_Q3_K, GATHER>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, slots, slices, part);
        case T_IQ4_XS: return launch_kq<T_IQ4_XS, GATHER>(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, slots, slices, part);
        default: return hipErrorInvalidValue;
    }
}

// Expert groups of these types with at most a tile for every CU: the staging kernel here too (us, staged / gemm_kr_kernel: Q6_K 13824
// values x 2928 rows, 2 experts, 144 pairs 97 / 122, 1280 x 800, 4 experts, 232 pairs 19.4 / 22.9; Q3_K 8960 x 280, 2 experts, 242 pairs 52.7 / 55.9;
// IQ4_XS 7936 x 1384, 4 experts, 396 pairs 65 / 76), whose tiles are 64 rows by 128 pairs.
// The number of tiles is known on the device only; ids drawn evenly pick n_as * (1 - e^(-pairs / n_as)) experts.
static bool kq_staged_groups(int wtype, int64_t N, int64_t n_as, int64_t pairs, int64_t cus) {
    if (wtype != T_Q6_K && wtype != T_Q3_K && wtype != T_IQ4_XS) return false;
    const float experts = (float)n_as, picked = experts * (1.f - std::exp(-(float)pairs / experts));
    return (picked + (float)pairs / (float)KqTile::BN) * (float)ceil_div(N, (int64_t)KqTile::BM) <= (float)cus;
}
int gemm_kq_moe_tile_tokens(int wtype, int64_t N, int64_t n_as, int64_t pairs, int compute_units) {
    return kq_staged_groups(wtype, N, n_as, pairs, compute_units > 0 ? compute_units : 256) ? KqTile::BN : gemm_kr_tile_tokens();
}

hipError_t launch_gemm_kq(int wtype, const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride,
                          int64_t M, float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather *rgp, int64_t n_as,
                          SplitK split) {
    if (M <= 0 || N <= 0 || n_as <= 0) return hipSuccess;
    if (!gemm_kq_type(wtype)) return hipErrorInvalidValue;
    const RowGather rg = rgp ? *rgp : RowGather{nullptr, nullptr, nullptr, 1, 1, 0};
    const GemmMats mats = one_gemm_mat(W, nb01, N, y, ldy);
    const int64_t cus = lim.compute_units > 0 ? lim.compute_units : 256;
    if (rg.perm && rg.tile_tokens == KqTile::BN) return launch_staged_type<true>(wtype, W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, 1, nullptr);
    if (rg.perm) return launch_gemm_kr(1, wtype, mats, K, ws, ws_stride, M, lim, st, rg, n_as, 1, nullptr);
    auto room = [&](int slices) {
        return slices <= 1 || (split.part && split.bytes >= (size_t)slices * (size_t)M * (size_t)N * sizeof(float) && (((uintptr_t)split.part) & 15) == 0);
    };
    KqPlan p = kq_plan(wtype, K, N, M, cus);
    // (unsplit for want of room: in the groups that more tokens of the same rows take, whose sums are added in the same order)
    if (!room(p.slices)) p = KqPlan{wtype == T_Q2_K || wtype == T_IQ4_XS ? (p.groups > 0 ? 2 : 0) : wtype != T_Q6_K && K > 8 * QK_K ? 2 : p.groups, 1};
    if (p.groups == 0) return launch_staged_type<false>(wtype, W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, 0, p.slices, split.part);
    return launch_gemm_kr(p.groups, wtype, mats, K, ws, ws_stride, M, lim, st, rg, n_as, p.slices, split.part);
}

// Members that run unsplit by themselves: the same bits, fewer launches and one set of tiles (us, ffn_gate + ffn_up, Q4_K
// of 4096 values x 14336 rows at 512 tokens, whose 896 tiles each leave a quarter of the second turn idle: 2 x 93.5 -> 164; wq + wk + wv of 1024
// values x 1024 + 256 + 256 rows at 128 tokens 36 -> 13).  A member is added up in the k groups that it has alone: all in the same number; or, Q4_K and
// Q5_K whose tiles together are more than the CUs, where one group is ahead (Q4_K 4352 values x 6424 rows twice at 244 tokens 50.3 us, in two 56.3), all in
// one, which walks the even super-blocks of those that alone have two and then the odd ones.  That walk fetches the lines that two super-blocks share
// twice: over 33 groups of two and three matrices 0.96 x the speed of the walk in order, which would add in another order (Q4_K 2816 values x 8213 rows
// twice at 171 tokens 32.1 / 34.0 us, 5120 x 3676 three times at 462 83.7 / 96.1).
// The k groups that a member alone runs in, 0: the staging kernel.  (IQ4_XS of 2 and 3 super-blocks: alone in the staging kernel, together
// faster in one launch; the same bits)
static int kq_own_groups(int wtype, int64_t K, int64_t N, int64_t n, int64_t cus) {
    return wtype == T_IQ4_XS && K < 4 * QK_K ? 1 : kq_plan(wtype, K, N, n, cus).groups;
}
// the k groups of the launch, 0: members that do not share one; even_odd is set where one group stands for two
static int kq_group_groups(int wtype, int64_t K, GemmMats &mats, int64_t n, int64_t cus) {
    const bool four = wtype == T_Q4_K || wtype == T_Q5_K;
    int64_t tiles = 0;
    int least = 2, most = 0;
    for (int i = 0; i < mats.count; i++) {
        const int own = kq_own_groups(wtype, K, mats.m[i].N, n, cus);
        mats.m[i].even_odd = four && own == 2;
        least = std::min(least, own);
        most = std::max(most, own);
        tiles += ceil_div(mats.m[i].N, (int64_t)128) * ceil_div(n, (int64_t)64);
    }
    if (least == 0 || (least != most && !four) || (least == 2 && (wtype == T_Q2_K || wtype == T_IQ4_XS))) return 0;
    if (least == 1 || (four && tiles > cus)) return 1;
    for (int i = 0; i < mats.count; i++) mats.m[i].even_odd = false;
    return 2;
}
bool gemm_kq_group_applicable(int wtype, int64_t K, const GemmMats &mats, int64_t n, int compute_units) {
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    if (mats.count < 2 || !gemm_kq_type(wtype)) return false;
    GemmMats t = mats;
    if (kq_group_groups(wtype, K, t, n, cus) == 0) return false;
    for (int i = 0; i < mats.count; i++) {
        const int64_t N = mats.m[i].N;
        if (!gemm_kq_supported(wtype, K, N, n, false) || kq_plan(wtype, K, N, n, cus).slices != 1) return false;
        if (gemm_kr_rows_in_reach(mats.m[i].nb01) < 32) return false;
    }
    return true;
}
hipError_t launch_gemm_kq_group(int wtype, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t n, const DeviceLimits &lim,
                                hipStream_t st) {
    GemmMats t = mats;
    const int groups = kq_group_groups(wtype, K, t, n, lim.compute_units > 0 ? lim.compute_units : 256);
    if (groups == 0) return hipErrorInvalidValue;
    return launch_gemm_kr(groups, wtype, t, K, ws, ws_stride, n, lim, st, RowGather{nullptr, nullptr, nullptr, 1, 1, 0}, 1, 1, nullptr);
}

}  // namespace chip
