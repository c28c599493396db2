// Prefill GEMM for gfx950 over K-quant weights (Q2_K .. Q6_K, IQ4_XS) and Q8_K activations: the batched form of
// lm_ggml_vec_dot_q2_K_q8_K .. _q6_K_q8_K, _iq4_xs_q8_K (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// This file holds the choice of the kernel and the staging kernel, which runs Q6_K where there is a tile for at most every CU;
// gemm_kr_kernel (gemm_kquant_rows.hip) runs everything else.
//
// Per 256-value super-block the reference forms sumi = sum_j sc_j * dot(q_j, a_j) with 8-bit signed scales per 16 values, and applies d
// and the activation scale once.  The integer scales are folded into the int8 MFMA operand, as the two signed bytes of (q - 32)*sc =
// 256*hi + lo, so both planes accumulate in the MFMA's own int32 accumulator over the 8 k-blocks of a super-block, sumi = 256*P0 + P1
// is exact, and the vector unit works once per super-block and output.
//
// Measured with these digits against base-64 digits of the product plus 4064 (16 instead of 10 vector instructions per four weights, and a
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

// Half h of a super-block holds, for l = 0..31, the elements 128h + 32b + l of k-blocks b = 0..3 as
//   low / high nibble of ql[64h + l] (b = 0 / 2) and of ql[64h + 32 + l] (b = 1 / 3), two more bits from
//   qh[32h + l] >> 2b, scale scales[8h + 2b + l/16]                       (reference ggml-quants.c:1695-1711)
// One staging item = (row, x) of a stage h: p = x / 2 picks the ql half (k-blocks p and p + 2), hf = x & 1 the 16 values
// l = 16*hf + [0,16) of both, which expand into one operand cell per digit plane and k-block.
struct Q6Item { u32x4 ql[2], qh[2], sc; uint32_t d; };
__device__ __forceinline__ void q6_fetch(Q6Item &r, const uint8_t *blk, int x) {
    const int p = x >> 1, hf = x & 1;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        r.ql[h] = *reinterpret_cast<const u32x4_a2 *>(blk + 64 * h + 32 * p + 16 * hf);
        r.qh[h] = *reinterpret_cast<const u32x4_a2 *>(blk + 128 + 32 * h + 16 * hf);
    }
    r.sc = *reinterpret_cast<const u32x4_a2 *>(blk + 192);
    r.d = *reinterpret_cast<const unsigned short *>(blk + 208);
}
// cell[plane][0: k-block p, 1: k-block p + 2]
__device__ __forceinline__ void q6_expand(u32x4 (&cell)[2][2], const Q6Item &r, int h, int x) {
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

constexpr int KQ_PRODUCERS = 4;               // staging waves per workgroup, one per SIMD

template <int WR, int WC>
struct KqCfg {
    static constexpr int NC = WR * WC;                             // MFMA waves
    static constexpr int NW = NC + KQ_PRODUCERS, NT = NW * 64;
    static constexpr int NPT = KQ_PRODUCERS * 64;                  // staging threads
    static constexpr int BM = 32 * WR;                             // weight rows per workgroup
    static constexpr int BN = 32 * KQ_TN * WC;                     // tokens per workgroup
    static constexpr int NPL = 2;                                  // int8 digit planes
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
template <int WR, int WC, int OCC>
__global__ __launch_bounds__((WR * WC + KQ_PRODUCERS) * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void gemm_kq_kernel(const uint8_t *__restrict__ W, size_t nb01, int64_t K, int64_t N, const uint8_t *__restrict__ ws,
                    size_t ws_stride, int64_t M, float *__restrict__ y, int64_t ldy, TileMap map, int slice_sb) {
    using C = KqCfg<WR, WC>;
    constexpr int TN = KQ_TN;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // split K: grid row s takes super-blocks sb0 .. of every row
    // and writes its partial tile to slice s of y
    int sb0 = 0, nstages = (int)(K / QK_K) * 2;
    if (slice_sb > 0) {
        sb0 = (int)blockIdx.y * slice_sb;
        nstages = 2 * min(slice_sb, (int)(K / QK_K) - sb0);
        y += (size_t)blockIdx.y * (size_t)M * (size_t)ldy;
    }
    const TileCoord tc = xcd_tile(blockIdx.x, map);
    if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;        // padding of the tile map
    const int64_t row_base = (int64_t)tc.row_tile * C::BM;
    const int64_t tok_base = (int64_t)tc.tok_tile * C::BN;
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
        struct Wts { Q6Item w[C::W_PER_T]; };
        Acts E, O;             // activations of an even / odd stage
        Wts W0, W1;            // weights of an even / odd super-block (both halves: every cache line is fetched once)
        // per-thread source addresses of stage 0 (they advance by a constant per stage / super-block)
        const uint8_t *wsrc[C::W_PER_T], *xsrc[C::X_PER_T];
#pragma unroll
        for (int i = 0; i < C::W_PER_T; i++) wsrc[i] = W + (size_t)min(row_base + ((pt + i * C::NPT) >> 2), N - 1) * nb01;
#pragma unroll
        for (int i = 0; i < C::X_PER_T; i++)
            xsrc[i] = ws + (size_t)min(tok_base + ((pt + i * C::NPT) >> 3), M - 1) * ws_stride + 16 * ((pt + i * C::NPT) & 7);
        // activation scale: thread t < BN for token t
        const uint8_t *ssrc = ws + (size_t)min(tok_base + min(pt, C::BN - 1), M - 1) * ws_stride;
        const int nsb = nstages >> 1;

        auto fetch_w = [&](Wts &R, int sb_wanted) {
            const int sb = min(sb_wanted, nsb - 1);
#pragma unroll
            for (int i = 0; i < C::W_PER_T; i++) q6_fetch(R.w[i], wsrc[i] + (size_t)(sb0 + sb) * BYTES_Q6_K, (pt + i * C::NPT) & 3);
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
                u32x4 cell[2][2];
                q6_expand(cell, RW.w[i], h, x);
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

    // once per super-block: fold the planes, out += d * float(256 * P0 + P1) * dx
    auto fold = [&](int sbp) {
        const uint8_t *sblk = lds + C::OFF_SBLK + (size_t)sbp * C::SBLK;
        const u32x4 *sp = reinterpret_cast<const u32x4 *>(sblk + C::OFF_SD) + (r0 + half * 16) / 4;
        const u32x4 s0 = sp[0], s1 = sp[1], s2 = sp[2], s3 = sp[3];
        const uint32_t sd[16] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w, s2.x, s2.y, s2.z, s2.w, s3.x, s3.y, s3.z, s3.w};
#pragma unroll
        for (int c = 0; c < TN; c++) {
            const float dx = reinterpret_cast<const float *>(sblk + C::OFF_SX)[n0 + c * 32 + l32];
#pragma unroll
            for (int v = 0; v < 16; v++) out[c][v] = __builtin_fmaf(h2f(sd[v]) * (float)((P[0][c][v] << 8) + P[1][c][v]), dx, out[c][v]);
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
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int64_t row = row_base + r0 + 8 * g + 4 * half;
            float *dst = y + (size_t)tok * ldy + row;
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
// Q6_K with a tile for at most every CU and more than a third as many, or on rows of fewer than 8 super-blocks: gemm_kq_kernel, whose
// staging waves expand a weight once for 128 tokens, in slices of its own (us, staged / gemm_kr_kernel: 14336 values x 4096 rows at 512 tokens
// 113 / 121, 201 tokens 66 / 73; 4096 x 4096 at 512 tokens 38.6 / 41.7; 1024 values x 4096 rows at 64 tokens 14.7 / 15.9).
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

static hipError_t launch_kq(const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride, int64_t M,
                            float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, int slices, float *part) {
    using C = KqCfg<2, 2>;                                               // 64 x 128, 4 + 4 waves
    const size_t lds_bytes = C::TOTAL;
    if ((int64_t)lds_bytes > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kq_kernel<2, 2, 2>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, lds_bytes, lim, grant); e != hipSuccess) return e;
    const TileMap map = make_tile_map(ceil_div(N, C::BM), ceil_div(M, C::BN), 32);      // 32 workgroups run on an XCD at a time
    const int slice_sb = slices > 1 ? (int)ceil_div(K / QK_K, (int64_t)slices) : 0;
    hipLaunchKernelGGL(kfn, dim3(map.grid, (unsigned)slices), dim3(C::NT), lds_bytes, st, (const uint8_t *)W, nb01, K, N,
                       (const uint8_t *)ws, ws_stride, M, slices > 1 ? part : y, slices > 1 ? N : ldy, map, slice_sb);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return slices > 1 ? launch_sum_slices(part, slices, M, N, y, ldy, st) : hipSuccess;
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
int gemm_kq_moe_tile_tokens() { return gemm_kr_tile_tokens(); }

hipError_t launch_gemm_kq(int wtype, const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride,
                          int64_t M, float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather *rgp, int64_t n_as,
                          SplitK split) {
    if (M <= 0 || N <= 0 || n_as <= 0) return hipSuccess;
    if (!gemm_kq_type(wtype)) return hipErrorInvalidValue;
    const RowGather rg = rgp ? *rgp : RowGather{nullptr, nullptr, nullptr, 1, 1, 0};
    if (rg.perm) return launch_gemm_kr(1, wtype, W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, 1, nullptr);
    const int64_t cus = lim.compute_units > 0 ? lim.compute_units : 256;
    auto room = [&](int slices) {
        return slices <= 1 || (split.part && split.bytes >= (size_t)slices * (size_t)M * (size_t)N * sizeof(float) && (((uintptr_t)split.part) & 15) == 0);
    };
    KrPlan p = kr_plan(K, N, M, cus);
    const bool staged = kq_staged(wtype, K, N, M, cus);
    if (wtype == T_Q6_K && (staged || !room(p.slices))) {                            // (the unsplit walk of few tiles: staged too)
        const int slices = staged ? kq_staged_slices(K, N, M, cus) : 1;
        return launch_kq(W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, room(slices) ? slices : 1, split.part);
    }
    if (!room(p.slices)) p = KrPlan{2, 1};
    return launch_gemm_kr(p.groups, wtype, W, nb01, K, N, ws, ws_stride, M, y, ldy, lim, st, rg, n_as, p.slices, split.part);
}

}  // namespace chip
