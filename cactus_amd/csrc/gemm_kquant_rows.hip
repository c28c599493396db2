// Prefill GEMM for gfx950 over K-quant weights (Q2_K .. Q6_K, IQ4_XS) and Q8_K activations: the batched form of
// lm_ggml_vec_dot_q2_K_q8_K .. _q6_K_q8_K, _iq4_xs_q8_K (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// Per 256-value super-block the reference forms two integers per (row, token), sumi = sum_j sc_j * dot(q_j, a_j) and (Q4_K, Q5_K,
// Q2_K) summ = sum_j m_j * bsum_j, and applies d, dmin and the activation scale once.  As in gemm_kquant.hip the integer sub-block
// scales ride in the int8 MFMA operand, as one or two digit planes whose products accumulate over the super-block in the MFMA's own int32
// registers, and summ is one fp16 MFMA (mins times the 16 block sums, exact):
//
//   Q4_K           sc = 8*sh + sl (3-bit digits): planes q*sh and q*sl (<= 105), sumi = 8*P0 + P1
//   Q5_K, Q6_K, IQ4_XS   the product v = q*sc, (q - 32)*sc, code*sc (16 bits) as 256*hi + lo with signed bytes, sumi = 256*P0 + P1
//   Q3_K           (4 - q)*sc in -128..124: one plane, sumi = -P0
//   Q2_K           q*sc <= 45: one plane, sumi = P0
//
// What is different is who expands.  There, staging waves write both planes of a 64 x 128 tile into LDS and every wave reads them back:
// twice the packed bytes times four in LDS traffic, two barriers per super-block, one stage of loads in flight.  Here a wave owns 32 weight
// rows and 64 tokens: it loads its rows' packed bytes in memory order, turns them round through a stretch of LDS of its own
// (no barrier), reads its MFMA lanes' quants back and expands them in registers between its MFMAs.  Only the activations are shared by the
// four waves of a k group (global_load_lds, double buffered), so a super-block needs one barrier and everything it waits for was
// requested a whole super-block earlier.
//
// Bound: the vector instructions and MFMAs of a SIMD do not overlap (403 and 34 per super-block and wave for Q4_K; 62 % + 40 % of the cycles
// by the counters, ffn_gate + ffn_up of 14336 rows x 4096 values at 512 tokens), LDS is 25 % busy, 2 % of it bank conflicts (Q6_K: 22 %).  Reading operands a step ahead took
// a quarter off the first form, in which every read was waited for at once; widening d and dmin once instead
// of in a half-rate v_fma_mix per output and full-rate v_bitop3 in place of v_and_or / v_bfi another 3 %.
// Measured against the staging kernel (Q4_K, Q5_K: the single-plane kernel) that ran these before, us for values x rows: Q4_K 512 tokens
// 4096 x 4096 40 -> 36.7, x 14336 105 -> 93.5, 14336 x 4096 110 -> 102, 32 tokens 14336 x 4096 38 -> 23; Q2_K 512 tokens 4096 x 14336
// 84 -> 68; Q5_K 512 tokens 14336 x 4096 139 -> 120; Q6_K 4096 x 14336 143 -> 121 at 512 tokens, 404 -> 316 at 1500.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include "kquant_rows_dev.h"
#include <type_traits>

namespace chip {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

namespace {

constexpr int KR_ROWS = 128;                  // weight rows per workgroup: four waves of 32

template <int WT, int TN, int KS>
struct KrCfg {
    using T = KR<WT>;
    static constexpr int NW = 4 * KS, NT = NW * 64;
    static constexpr int BN = 32 * TN;                                    // tokens per workgroup
    static constexpr int NLD = (32 * T::NCH + 63) / 64;                   // chunk loads of a lane per super-block
    static constexpr int B_PER_W = BN / 16;                               // direct loads of a wave per super-block (four tokens each)
    static constexpr size_t RAW = (size_t)NLD * 1024;                     // per wave: its 32 rows of one super-block, whole loads
    static constexpr size_t OFF_B = RAW * NW;                             // [buffer][k group] activations, [token][16 cells] swizzled
    static constexpr size_t B_BYTES = (size_t)BN * 256;
    // What the fold reads has four buffers: a wave folds super-block j behind the barrier that follows its products, while a faster
    // one already writes the values of super-block j + 2 in front of the next barrier.
    static constexpr size_t OFF_FB = OFF_B + 2 * KS * B_BYTES;            // [j % 4][k group] fp16 cells [k-half][token]: the 16 bsums
    static constexpr size_t FB_BYTES = T::NF16 > 0 ? (size_t)BN * 32 : 0;
    static constexpr size_t OFF_SX = OFF_FB + 4 * KS * FB_BYTES;          // [j % 4][k group] f32 [token]: activation scale
    static constexpr size_t OFF_ROW = OFF_SX + 4 * KS * (size_t)BN * 4;   // i32 [token]: output row (expert groups)
    static constexpr size_t TOTAL = OFF_ROW + (size_t)BN * 4;
    // EVEN_ODD: as many of a lane's 16 TN sums as leave room for two workgroups a CU wait here, [wave][sum][lane]; the rest in registers
    static constexpr int ROOM = (80 * 1024 - (int)TOTAL) / (NW * 256), WAIT = ROOM < 0 ? 0 : ROOM < 16 * TN ? ROOM : 16 * TN;
    static constexpr size_t TOTAL_EVEN_ODD = TOTAL + (size_t)WAIT * NW * 256;
    // the other k groups' partial outputs take the place of the operands at the end
    static_assert((size_t)(KS - 1) * 4 * TN * 16 * 256 <= OFF_SX, "partial outputs lie in front of the output rows");
};

__device__ __forceinline__ void kr_load16_into_lds(const uint8_t *base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory");
}
__device__ __forceinline__ void kr_load16_into_lds(const uint8_t *src, uint32_t lds_addr) {
    // M0 = LDS byte address of the wave's 1 KB destination; lane i's 16 bytes land at M0 + 16 i.  Inline assembly so that
    // the compiler does not make every later LDS read wait for it; the kernel waits by hand in front of the barrier.
    // Nothing else in the kernel may use M0 (no dynamic register indexing).
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_addr) : "memory");
}

// EVEN_ODD: matrices with even_odd set are walked over their even super-blocks and then over the odd ones; in between the sums wait in LDS and registers
// (in y they took 11 to 17 us of a launch of 30 to 130).
template <int WT, int TN, int KS, int OCC, bool GATHER, bool EVEN_ODD>
__global__ __launch_bounds__(4 * KS * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void gemm_kr_kernel(GemmMats mats, int64_t K, const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M, TileMap map, RowGather rg,
                    int slice_sb) {
    using T = KR<WT>;
    using C = KrCfg<WT, TN, KS>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, wr = wave & 3;                            // k group, row tile
    const int gt = tid & 255;                                            // thread of the k group
    int sb0 = 0, nsb = (int)(K / QK_K);
    if (!GATHER && slice_sb > 0) {
        sb0 = (int)blockIdx.y * slice_sb;
        nsb = min(slice_sb, nsb - sb0);
    }
    TileCoord tc;
    int32_t entry = 0;
    if constexpr (GATHER) {
        if (!gather_tile<C::BN>(rg, map, entry, tc.row_tile)) return;
        tc.tok_tile = 0;
    } else {
        tc = xcd_tile(blockIdx.x, map);
        if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;        // padding of the tile map
    }
    const GemmMat mat = GATHER ? mats.m[0] : pick_gemm_mat(mats, tc.row_tile);
    const int evens = EVEN_ODD && mat.even_odd ? (nsb + 1) / 2 : nsb;     // super-blocks in front of the turn to the odd ones
    auto nth = [&](int i) {                                              // the i-th super-block of the walk (past the end: the last)
        i = min(i, nsb - 1);
        if constexpr (EVEN_ODD) return evens == nsb ? i : i < evens ? 2 * i : 2 * (i - evens) + 1;
        return i;
    };
    const int64_t N = mat.N, ldy = mat.ldy;
    const size_t nb01 = mat.nb01;
    float *__restrict__ y = mat.y;
    if (!GATHER && slice_sb > 0) y += (size_t)blockIdx.y * (size_t)M * (size_t)ldy;
    size_t w_offset;
    const GatherView gv = resolve_gather<GATHER>(rg, entry, w_offset, M);
    const uint8_t *__restrict__ W = mat.W + w_offset;
    const int64_t row_base = (int64_t)tc.row_tile * KR_ROWS + wr * 32;
    const int64_t tok_base = (int64_t)(GATHER ? gv.tok_tile : tc.tok_tile) * C::BN;
    if (tok_base >= M) return;
    const int tokens = (int)min((int64_t)C::BN, M - tok_base);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const size_t off_d = q8_K_off_d(K), off_bs = q8_K_off_bsums(K);
    const int half = lane >> 5, l32 = lane & 31;

    // ---- weights: the wave's own 32 rows, chunk by chunk in memory order, through registers into its own stretch of LDS ----
    const int64_t row_c = min(row_base, N - 1);
    const uint8_t *wbase = W + (size_t)row_c * nb01 + (size_t)sb0 * T::BYTES;
    uint32_t woff[C::NLD];
#pragma unroll
    for (int t = 0; t < C::NLD; t++) {
        const int i = min(lane + 64 * t, 32 * T::NCH - 1), r = i / T::NCH, c = i % T::NCH;
        woff[t] = (uint32_t)(min(row_base + r, N - 1) - row_c) * (uint32_t)nb01 + (uint32_t)(c == T::NCH - 1 ? T::BYTES - 16 : 16 * c);
    }
    u32x4 *const raw_lds = reinterpret_cast<u32x4 *>(lds + C::RAW * wave);
    u32x4 raw[C::NLD];
    auto fetch_w = [&](int sb_wanted) {
        const uint8_t *p = wbase + (size_t)nth(sb_wanted) * T::BYTES;
#pragma unroll
        for (int t = 0; t < C::NLD; t++) raw[t] = *reinterpret_cast<const typename T::chunk_t *>(p + woff[t]);
    };
    auto commit_w = [&]() {
#pragma unroll
        for (int t = 0; t < C::NLD; t++) raw_lds[lane + 64 * t] = raw[t];
    };

    // ---- activations: the k group's BN tokens of its super-block straight into LDS, 256-byte rows of 16 swizzled cells ----
    // (a plain tile's tokens lie side by side: one scalar base and 32-bit offsets)
    const uint8_t *const act0 = ws + (size_t)(GATHER ? 0 : tok_base) * ws_stride + (size_t)sb0 * QK_K;
    const uint8_t *bsrc[GATHER ? C::B_PER_W : 1];
    uint32_t boff[GATHER ? 1 : C::B_PER_W];
#pragma unroll
    for (int j = 0; j < C::B_PER_W; j++) {
        const int t = (wr * C::B_PER_W + j) * 4 + (lane >> 4);
        const uint32_t cell = 16u * (uint32_t)((lane & 15) ^ (t & 15));
        if constexpr (GATHER) bsrc[j] = act0 + (size_t)gv.act_row(min(tok_base + t, M - 1)) * ws_stride + cell;
        else boff[j] = (uint32_t)min(t, tokens - 1) * (uint32_t)ws_stride + cell;
    }
    auto issue_x = [&](int sb_wanted, int buf) {
        const size_t o = (size_t)nth(sb_wanted) * QK_K;
        const uint32_t dst = lds0 + (uint32_t)(C::OFF_B + (size_t)(buf * KS + grp) * C::B_BYTES) + (uint32_t)(wr * C::B_PER_W) * 1024u;
#pragma unroll
        for (int j = 0; j < C::B_PER_W; j++) {
            const uint32_t d = __builtin_amdgcn_readfirstlane(dst + (uint32_t)j * 1024u);
            if constexpr (GATHER) kr_load16_into_lds(bsrc[j] + o, d);
            else kr_load16_into_lds(act0 + o, boff[j], d);
        }
    };
    // activation scale: thread t < BN of the k group for token t; block sums: thread t < 2*BN for token t/2, k-half t&1
    const uint8_t *ssrc = ws + (size_t)gv.act_row(min(tok_base + min(gt, C::BN - 1), M - 1)) * ws_stride + off_d + (size_t)sb0 * 4;
    const uint8_t *bssrc = ws + (size_t)gv.act_row(min(tok_base + min(gt >> 1, C::BN - 1), M - 1)) * ws_stride + off_bs + 16 * (gt & 1) + (size_t)sb0 * 32;
    float xs;
    u32x4 bs;
    auto fetch_s = [&](int sb_wanted) {
        const int sb = nth(sb_wanted);
        xs = reinterpret_cast<const float *>(ssrc)[sb];
        if constexpr (T::NF16 > 0) bs = *reinterpret_cast<const u32x4 *>(bssrc + (size_t)sb * 32);
    };
    auto commit_s = [&](int it) {
        const int q = (it & 3) * KS + grp;
        if (gt < C::BN) reinterpret_cast<float *>(lds + C::OFF_SX)[q * C::BN + gt] = xs;
        if constexpr (T::NF16 > 0)
            if (gt < 2 * C::BN)
                *reinterpret_cast<u32x4 *>(lds + C::OFF_FB + (size_t)q * C::FB_BYTES + (size_t)((gt & 1) * C::BN + (gt >> 1)) * 16) = i16x8_to_f16(bs);
    };

    float out[TN][16];
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
        for (int v = 0; v < 16; v++) out[c][v] = 0.f;

    // at the turn to the odd super-blocks
    float kept[EVEN_ODD ? 16 * TN - C::WAIT : 1] = {};
    float *const waiting = reinterpret_cast<float *>(lds + C::TOTAL) + wave * C::WAIT * 64 + lane;
    auto turn = [&]() {
#pragma unroll
        for (int i = 0; i < 16 * TN; i++) {
            float &o = out[i / 16][i % 16];
            if (i < C::WAIT) waiting[i * 64] = o;
            else kept[i - C::WAIT] = o;
            o = 0.f;
        }
    };

    // This wave's 32 rows against the first 32*NTL of the tile's tokens.  Activations are the MFMA's first operand: register v of tile c
    // is token 32 c + 8 (v / 4) + 4 half + v % 4, the lane's l32 its row.
    //
    // Super-block it * KS + grp in iteration it, in four steps of two k-blocks.  Step Q multiplies what the step before it read and
    // expanded, reads the operands of step Q + 1 and expands its weights between its own MFMAs.  The weights of the next iteration
    // travel in registers and take the place of the current ones in LDS in step 3, when those have all been read; the next activations
    // go straight into the other buffer.  Both were requested an iteration before the one barrier that makes them visible; behind it
    // the fold runs together with the reads and the expansion of the next super-block's step 0.
    constexpr int WAIT0 = 0x0F70;                                          // s_waitcnt vmcnt(0)
    const int nit = (nsb + KS - 1) / KS;
    const u32x4 *const row_lds = raw_lds + l32 * T::NCH;
    const uint32_t b_lane = (uint32_t)l32 * 256u + 16u * (uint32_t)(half ^ (l32 & 15));
    auto walk = [&](auto ntl_tag) {
        constexpr int NTL = decltype(ntl_tag)::value;
        typename T::Hdr h;
        typename T::Raw r1;
        u32x4 cc[2][T::NPL], cn[2][T::NPL], bc[2][NTL], bn[2][NTL];
        i32x16 P[T::NPL][NTL];
        auto load_b = [&](u32x4 (&b)[2][NTL], int buf, int ka, int kb) {
            const uint8_t *p = lds + (C::OFF_B + (size_t)(buf * KS + grp) * C::B_BYTES);
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int c = 0; c < NTL; c++) b[e][c] = *reinterpret_cast<const u32x4 *>(p + (b_lane ^ (uint32_t)(32 * (e ? kb : ka))) + c * 8192);
        };
        auto multiply = [&](auto first_tag) {
            constexpr bool first = decltype(first_tag)::value;
            const i32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int c = 0; c < NTL; c++)
#pragma unroll
                    for (int pl = 0; pl < T::NPL; pl++)
                        P[pl][c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, bc[e][c]), __builtin_bit_cast(i32x4, cc[e][pl]),
                                                                         (first && e == 0) ? zero : P[pl][c], 0, 0, 0);
        };
        auto step = [&](auto q_tag, int buf) {
            constexpr int Q = decltype(q_tag)::value;
            typename T::Raw r2;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (Q < 3) load_b(bn, buf, kr_k_block<T>((Q + 1) >> 1, (Q + 1) & 1, 0), kr_k_block<T>((Q + 1) >> 1, (Q + 1) & 1, 1));
            if constexpr (Q < 2) r2 = T::load(row_lds, 1, Q, half);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (Q < 3) T::expand(r1, h, (Q + 1) >> 1, (Q + 1) & 1, half, cn);
            multiply(std::integral_constant<bool, Q == 0>{});
            if constexpr (Q < 3) {
                constexpr int MF = 2 * NTL * T::NPL;
#pragma unroll
                for (int i = 0; i < MF; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 96 / MF, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 2; e++) {
#pragma unroll
                    for (int pl = 0; pl < T::NPL; pl++) cc[e][pl] = cn[e][pl];
#pragma unroll
                    for (int c = 0; c < NTL; c++) bc[e][c] = bn[e][c];
                }
            }
            if constexpr (Q < 2) r1 = r2;
        };
        // reads step 0 of the super-block in `buf`; its weights are expanded behind the fold, whose registers are free then
        typename T::Raw r0;
        auto first_operands = [&](int buf) {
            h = T::hdr(row_lds, half);
            r0 = T::load(row_lds, 0, 0, half);
            r1 = T::load(row_lds, 0, 1, half);
            load_b(bc, buf, kr_k_block<T>(0, 0, 0), kr_k_block<T>(0, 0, 1));
        };

        issue_x(grp, 0);
        fetch_w(grp);
        fetch_s(grp);
        if constexpr (GATHER)
            if (tid < C::BN) reinterpret_cast<int32_t *>(lds + C::OFF_ROW)[tid] = gv.list[tok_base + min(tid, tokens - 1)];
        commit_w();
        commit_s(0);
        __builtin_amdgcn_s_waitcnt(WAIT0);
        __syncthreads();
        fetch_w(grp + KS);
        fetch_s(grp + KS);
        first_operands(0);
        T::expand(r0, h, 0, 0, half, cc);
        auto iteration = [&](int it, auto last_tag) {
            constexpr bool last = decltype(last_tag)::value;                  // nothing left to request
            const int buf = it & 1, sb = it * KS + grp, q4 = (it & 3) * KS + grp;
            if constexpr (!last) issue_x(sb + KS, buf ^ 1);
            step(std::integral_constant<int, 0>{}, buf);
            step(std::integral_constant<int, 1>{}, buf);
            step(std::integral_constant<int, 2>{}, buf);
            step(std::integral_constant<int, 3>{}, buf);
            float d = h2f(T::scales(h)), dmin = h2f(T::scales(h) >> 16);
            asm volatile("" : "+v"(d), "+v"(dmin));                        // widened once: as halves they would make every multiply-add a half-rate mixed one
            f16x8 fa[T::NF16 > 0 ? T::NF16 : 1];
#pragma unroll
            for (int f = 0; f < T::NF16; f++) fa[f] = __builtin_bit_cast(f16x8, T::f16_cell(h, f, half));
            if constexpr (!last) {
                commit_w();
                commit_s(it + 1);
                __builtin_amdgcn_s_waitcnt(WAIT0);
                __syncthreads();
                fetch_w(sb + 2 * KS);
                fetch_s(sb + 2 * KS);
                first_operands(buf ^ 1);
            }
            // fold: out += dx * (d * float(sumi) - dmin * summ); the last iteration may lie past a k group's end
#pragma unroll
            for (int c = 0; c < NTL; c++) {
                f32x16 F[T::NF16 > 0 ? T::NF16 : 1];
                if constexpr (T::NF16 > 0) {
                    const f16x8 fb = *reinterpret_cast<const f16x8 *>(lds + C::OFF_FB + (size_t)q4 * C::FB_BYTES + (size_t)(half * C::BN + c * 32 + l32) * 16);
                    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int f = 0; f < T::NF16; f++) F[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb, fa[f], zero, 0, 0, 0);
                }
                const float *sx = reinterpret_cast<const float *>(lds + C::OFF_SX) + q4 * C::BN + c * 32 + 4 * half;
                float dxv[16];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float4 dx = *reinterpret_cast<const float4 *>(sx + 8 * g);
                    dxv[4 * g] = dx.x; dxv[4 * g + 1] = dx.y; dxv[4 * g + 2] = dx.z; dxv[4 * g + 3] = dx.w;
                }
                if (KS == 1 || sb < nsb) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    float f[2] = {0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < T::NF16; j++) f[j] = F[j][v];
                    out[c][v] = __builtin_fmaf(T::value(P[0][c][v], P[T::NPL - 1][c][v], f, d, dmin), dxv[v], out[c][v]);
                }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!last) T::expand(r0, h, 0, 0, half, cc);
        };
        int it = 0;
        if constexpr (EVEN_ODD) {
            for (; it < evens && it + 1 < nit; it++) iteration(it, std::false_type{});
            if (evens < nsb) turn();
        }
        for (; it + 1 < nit; it++) iteration(it, std::false_type{});
        iteration(nit - 1, std::true_type{});
        __syncthreads();
    };
    if (TN > 1 && tokens <= 32) walk(std::integral_constant<int, 1>{});
    else walk(std::integral_constant<int, TN>{});

    // the k groups' partial sums meet in LDS and are added in order
    if constexpr (KS > 1) {
        float *part = reinterpret_cast<float *>(lds);
        if (grp > 0) {
#pragma unroll
            for (int c = 0; c < TN; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) part[(((grp - 1) * 4 + wr) * TN * 16 + c * 16 + v) * 64 + lane] = out[c][v];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 1; g < KS; g++)
#pragma unroll
            for (int c = 0; c < TN; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) out[c][v] += part[(((g - 1) * 4 + wr) * TN * 16 + c * 16 + v) * 64 + lane];
    }
    if constexpr (EVEN_ODD)
        if (evens < nsb)
#pragma unroll
            for (int i = 0; i < 16 * TN; i++) out[i / 16][i % 16] += i < C::WAIT ? waiting[i * 64] : kept[i < C::WAIT ? 0 : i - C::WAIT];
    const int64_t row = row_base + l32;
    if (row >= N) return;
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int t0 = c * 32 + 8 * g + 4 * half;
            int32_t orow[4];
            if constexpr (GATHER) *reinterpret_cast<u32x4 *>(orow) = *reinterpret_cast<const u32x4 *>(lds + C::OFF_ROW + t0 * 4);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (t0 + e < tokens) y[(size_t)(GATHER ? orow[e] : tok_base + t0 + e) * ldy + row] = out[c][4 * g + e];
        }
}

template <int WT, int TN, int KS, int OCC, bool GATHER, bool EVEN_ODD = false>
hipError_t launch_kr(GemmMats mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim, hipStream_t st,
                     const RowGather &rg, int64_t slots, int slices, float *part) {
    using C = KrCfg<WT, TN, KS>;
    constexpr size_t LDS = EVEN_ODD ? C::TOTAL_EVEN_ODD : C::TOTAL;
    if ((int64_t)LDS > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kr_kernel<WT, TN, KS, OCC, GATHER, EVEN_ODD>;
    static LdsGrant grant;                                               // one per kernel instantiation
    if (hipError_t e = grant_dynamic_lds(kfn, LDS, lim, grant); e != hipSuccess) return e;
    const int per_cu = (int)(160 * 1024 / LDS) > 0 ? (int)(160 * 1024 / LDS) : 1;
    const int64_t row_tiles = number_row_tiles(mats, KR_ROWS);
    if constexpr (GATHER) {
        const TileMap map = make_tile_map(row_tiles, 1, 32 * per_cu);
        hipLaunchKernelGGL(kfn, gather_grid(map, slots, C::NT), dim3(C::NT), LDS, st, mats, K, (const uint8_t *)ws, ws_stride, M, map, rg, 0);
        return hipGetLastError();
    } else {
        const TileMap map = make_tile_map(row_tiles, ceil_div(M, C::BN), 32 * per_cu);
        const GemmMat out = mats.m[0];
        const int slice_sb = slices > 1 ? (int)ceil_div(K / QK_K, (int64_t)slices) : 0;
        if (slices > 1) { mats.m[0].y = part; mats.m[0].ldy = out.N; }                  // (one matrix)
        hipLaunchKernelGGL(kfn, dim3(map.grid, (unsigned)slices), dim3(C::NT), LDS, st, mats, K, (const uint8_t *)ws, ws_stride, M, map, rg, slice_sb);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        return slices > 1 ? launch_sum_slices(part, slices, M, out.N, out.y, out.ldy, st, WT == T_Q2_K || WT == T_IQ4_XS) : hipSuccess;
    }
}

template <int WT>
hipError_t launch_kr_groups(int groups, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim,
                            hipStream_t st, const RowGather &rg, int64_t slots, int slices, float *part) {
    if (rg.perm) return launch_kr<WT, 2, 1, 2, true>(mats, K, ws, ws_stride, M, lim, st, rg, slots, 1, nullptr);   // expert groups
    if (groups == 2) return launch_kr<WT, 2, 2, 2, false>(mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
    if constexpr (WT == T_Q4_K || WT == T_Q5_K)
        for (int i = 0; i < mats.count; i++)
            if (mats.m[i].even_odd) return launch_kr<WT, 2, 1, 2, false, true>(mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
    return launch_kr<WT, 2, 1, 2, false>(mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
}

}  // namespace

int gemm_kr_tile_tokens() { return KrCfg<T_Q4_K, 2, 1>::BN; }

// A lane reaches its rows by 32-bit offsets from the first of the wave's 32: how many rows of this stride they cover (32: any tile).
int64_t gemm_kr_rows_in_reach(size_t nb01) {
    const size_t more = (size_t)(0xffffffffu - BYTES_Q6_K) / nb01;
    return more < 31 ? (int64_t)more + 1 : 32;
}

hipError_t launch_gemm_kr(int groups, int wtype, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M,
                          const DeviceLimits &lim, hipStream_t st, const RowGather &rg, int64_t slots, int slices, float *part) {
    // rows more than 138 MB apart (a view of every n-th row, say): a launch for every stretch within reach
    if (const int64_t reach = gemm_kr_rows_in_reach(mats.m[0].nb01), N = mats.m[0].N; reach < 32 && reach < N) {
        for (int64_t r = 0; r < N; r += reach) {
            GemmMats t = mats;                                           // (one matrix: gemm_kq_group_applicable)
            t.m[0].W += (size_t)r * t.m[0].nb01;
            t.m[0].y += r;
            t.m[0].N = reach < N - r ? reach : N - r;
            if (hipError_t e = launch_gemm_kr(groups, wtype, t, K, ws, ws_stride, M, lim, st, rg, slots, slices, part); e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    switch (wtype) {
        case T_Q4_K: return launch_kr_groups<T_Q4_K>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        case T_Q5_K: return launch_kr_groups<T_Q5_K>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        case T_Q6_K: return launch_kr_groups<T_Q6_K>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        case T_Q3_K: return launch_kr_groups<T_Q3_K>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        case T_Q2_K: return launch_kr_groups<T_Q2_K>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        case T_IQ4_XS: return launch_kr_groups<T_IQ4_XS>(groups, mats, K, ws, ws_stride, M, lim, st, rg, slots, slices, part);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace chip
