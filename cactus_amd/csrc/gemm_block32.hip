// Prefill GEMM for gfx950 over weights in 32-value blocks with one fp16 scale each (Q4_0, Q8_0, Q5_0, IQ4_NL; Q4_1 and
// Q5_1 with a minimum on top) and Q8_0 / Q8_1 activations: Y[t][r] = sum_b dw[r][b] * dx[t][b] * isum[t][r][b], the batched form of lm_ggml_vec_dot_q4_0_q8_0,
// _q8_0_q8_0, _q5_0_q8_0 and _iq4_nl_q8_0 (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// Structure
//   * One v_mfma_i32_32x32x32_i8 multiplies a 32-row x 32-k weight tile by a 32-k x 32-token activation tile:
//     its K extent is exactly one 32-value quantization block, so each of the 1024 int32 results is one
//     per-block integer sum isum[t][r][b], bit-exact.
//   * Weight tiles are staged through LDS once per workgroup and k-stage: a block's packed quants are expanded into
//     two 16-byte cells of signed int8 (elements 0..15 and 16..31), possibly times a power of two that is taken
//     back exactly in the epilogue (Q4_0: 16 * (nib - 8), Q5_0: 8 * (q - 16); IQ4_NL: the code point; Q8_0: as is);
//     activations arrive as int8 from the split workspace layout.
//   * Per-block scales are applied in fp32 after the integer accumulate.  The MFMA's C input is a register
//     vector holding the bit pattern of 12582912.0f (1.5 * 2^23): adding |isum| < 2^22 to those bits gives the
//     bits of the float 12582912 + isum, so the accumulator can be used as a float with no conversion.  Then
//         t   = fma(acc_as_float, dx, -12582912 * dx)      exactly round(isum * dx): 12582912*dx is exact
//                                                           because dx comes from fp16 (11-bit significand)
//         out = fma(t, dw, out)                            dw widened to fp32 exactly
//     i.e. two VALU operations per integer sum, 32 per MFMA.  That VALU work, not the matrix pipe, bounds this
//     kernel: an MFMA occupies the matrix unit for 32 cycles; the 32 fp32 operations, which read the MFMA's result
//     registers, take 134 - 144 cycles per SIMD with two to four waves (measured in a register-only loop).
//   * Q4_1 and Q5_1 add m * s per block (the weight block's minimum times the activation block's d * sum, the s of
//     block_q8_1).  Both factors are fp16 numbers, so sum_b m[r][b] * s[t][b] over the 4 blocks of a stage is one
//     v_mfma_f32_32x32x8f16 that adds straight into the fp32 accumulators: no vector work.
//   * A workgroup is WR x WC waves, each wave owns TM x TN MFMA tiles (32*TM rows x 32*TN tokens); LDS is
//     double buffered over stages of KB = 4 blocks with one barrier per stage.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace chip {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int GEMM_KB = 4;                    // 32-value blocks per LDS stage
constexpr float MAGIC_F = 12582912.f;         // 1.5 * 2^23
constexpr int MAGIC_I = 0x4B400000;

// How a weight type's block becomes two MFMA operand cells.  MULT is the power of two the cells carry on top of the
// quant (taken back through the activation scale, exactly); MULT * |isum| stays below 2^22 for every type.
template <int WT> struct Blk32;

template <> struct Blk32<T_Q4_0> {
    static constexpr int BYTES = BYTES_Q4_0;
    static constexpr bool HAS_MIN = false;
    static constexpr float INV_MULT = 1.f / 16.f;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) { r.q = *reinterpret_cast<const u32x4_a2 *>(p + 2); }
    // a nibble moved to the high half of its byte with its top bit flipped is 16 * (nibble - 8) as a signed byte
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = ((r.q[i] << 4) & 0xf0f0f0f0u) ^ 0x80808080u;
            hi[i] = (r.q[i] & 0xf0f0f0f0u) ^ 0x80808080u;
        }
    }
};

template <> struct Blk32<T_IQ4_NL> {
    static constexpr int BYTES = BYTES_IQ4_NL;
    static constexpr bool HAS_MIN = false;
    static constexpr float INV_MULT = 1.f;
    using Raw = Blk32<T_Q4_0>::Raw;
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) { Blk32<T_Q4_0>::fetch(r, p); }
    // four code indices (one per byte, 0..15) -> four code points of kvalues_iq4nl (reference ggml-common.h), through
    // two byte permutes of the 16-entry table
    __device__ static __forceinline__ uint32_t lookup4(uint32_t idx) {
        constexpr uint32_t T0 = 0xbfad9881u, T1 = 0xf6eaddcfu, T2 = 0x26190d01u, T3 = 0x71594535u;
        const uint32_t sel = idx & 0x07070707u;
        const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
        const uint32_t m = ((idx >> 3) & 0x01010101u) * 0xffu;
        return (lo & ~m) | (hi & m);
    }
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = lookup4(r.q[i] & 0x0f0f0f0fu);
            hi[i] = lookup4((r.q[i] >> 4) & 0x0f0f0f0fu);
        }
    }
};

template <> struct Blk32<T_Q8_0> {
    static constexpr int BYTES = BYTES_Q8_0;
    static constexpr bool HAS_MIN = false;
    static constexpr float INV_MULT = 1.f;
    struct Raw { u32x4 lo, hi; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) {
        r.lo = *reinterpret_cast<const u32x4_a2 *>(p + 2);
        r.hi = *reinterpret_cast<const u32x4_a2 *>(p + 18);
    }
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) { lo = r.lo; hi = r.hi; }
};

template <> struct Blk32<T_Q5_0> {
    static constexpr int BYTES = BYTES_Q5_0;
    static constexpr bool HAS_MIN = false;
    static constexpr float INV_MULT = 1.f / 8.f;
    struct Raw { u32x4 q; uint32_t qh; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) {
        r.qh = *reinterpret_cast<const u32_a2 *>(p + 2);
        r.q = *reinterpret_cast<const u32x4_a2 *>(p + 6);
    }
    // element j < 16: low nibble of qs[j] with bit j of qh on top, element 16 + j: high nibble with bit 16 + j
    // (reference ggml-quants.c:290-310).  The cell byte is 8 * (q - 16): q << 3 with the top bit flipped.
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // 4 bits -> bit 0 of each byte: bit k lands at 7k + k = 8k
            const uint32_t bl = (((r.qh >> (4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u;
            const uint32_t bh = (((r.qh >> (16 + 4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u;
            lo[i] = (((r.q[i] << 3) & 0x78787878u) | (bl << 7)) ^ 0x80808080u;
            hi[i] = (((r.q[i] >> 1) & 0x78787878u) | (bh << 7)) ^ 0x80808080u;
        }
    }
};

// Q4_1 / Q5_1: unsigned quants, block = d, m (fp16), [qh,] qs; value = d * q + m
template <> struct Blk32<T_Q4_1> {
    static constexpr int BYTES = BYTES_Q4_1;
    static constexpr bool HAS_MIN = true;
    static constexpr float INV_MULT = 1.f / 8.f;
    struct Raw { u32x4 q; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) { r.q = *reinterpret_cast<const u32x4_a4 *>(p + 4); }
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) {      // 8 * nibble, 0..120
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = (r.q[i] << 3) & 0x78787878u;
            hi[i] = (r.q[i] >> 1) & 0x78787878u;
        }
    }
};

template <> struct Blk32<T_Q5_1> {
    static constexpr int BYTES = BYTES_Q5_1;
    static constexpr bool HAS_MIN = true;
    static constexpr float INV_MULT = 1.f / 4.f;
    struct Raw { u32x4 q; uint32_t qh; };
    __device__ static __forceinline__ void fetch(Raw &r, const uint8_t *p) {
        r.qh = *reinterpret_cast<const uint32_t *>(p + 4);
        r.q = *reinterpret_cast<const u32x4_a4 *>(p + 8);
    }
    __device__ static __forceinline__ void emit(const Raw &r, u32x4 &lo, u32x4 &hi) {      // 4 * q, 0..124
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t bl = (((r.qh >> (4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u;
            const uint32_t bh = (((r.qh >> (16 + 4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u;
            lo[i] = ((r.q[i] << 2) & 0x3c3c3c3cu) | (bl << 6);
            hi[i] = ((r.q[i] >> 2) & 0x3c3c3c3cu) | (bh << 6);
        }
    }
};

// ---- how the operands travel and how a wave orders its work ----
//   * Quantized activations and their scales go from the workspace into LDS with global_load_lds_dwordx4: no staging
//     registers, no ds_write, no vector instructions.  A token's 128 bytes of a stage are one LDS row of 8 cells; cell c of
//     token t sits in slot c ^ ((t >> 1) & 7), so the 16 lanes that read one cell index of 16 consecutive tokens hit 16
//     different bank groups (the lane that fills a slot fetches the matching cell).  The four fp32 scales of a token and
//     stage are one more cell.
//   * Weights pass through registers (their 18- to 34-byte blocks must be expanded to int8 cells); they are fetched
//     two stages ahead and expanded one stage ahead, so a load has a whole stage to arrive.  The weight scales are
//     widened to fp32 on the way into LDS: a mixed-precision FMA that reads them as fp16 issues at a lower rate than a
//     plain one (measured: 16 + 16 plain FMAs behind an MFMA 56 - 60 ns per SIMD, with the second 16 mixed 67 - 80 ns).
//   * Inside a stage the MFMA of tile i + 1 is issued before the 32 scaling operations of tile i, across k-blocks too,
//     so one wave keeps the vector unit busy by itself and two waves per SIMD are enough; the stage loop is unrolled by
//     two so that every LDS address is a register plus an immediate.
//   * The power of two that the weight cells carry is taken back once, in the epilogue (exact), not per stage.
// LDS cells: [k-block][half][row] 16-byte cells for the weights (exactly what one lane feeds the MFMA: row = lane % 32,
// half = lane / 32), each plane padded by two cells: the threads that expand one stage walk the planes fastest, and a
// plane stride that is 2 mod 16 cells puts 16 consecutive writers on 16 different bank groups.
template <int TM, int TN, int WR, int WC, bool HAS_MIN>
struct DirectCfg {
    static constexpr int NW = WR * WC, NT = NW * 64;
    static constexpr int BM = 32 * TM * WR, BN = 32 * TN * WC;
    static constexpr int A_PLANE = BM + 2;                                        // cells
    static constexpr size_t OFF_A = 0;
    static constexpr size_t OFF_B = OFF_A + (size_t)GEMM_KB * 2 * A_PLANE * 16;   // [token][8 cells], swizzled
    static constexpr size_t OFF_SX = OFF_B + (size_t)BN * 128;                    // [token][4 floats]
    static constexpr size_t OFF_SW = OFF_SX + (size_t)BN * 16;                    // fp32 [KB][BM], permuted per 32 rows
    // plane b of the weight scales starts 8 * (b & 1) + 32 * (b >> 1) floats late: the 64 lanes that expand 16 rows x 4
    // k-blocks then write to 64 different banks (a row's position inside its 32-row group is 0..7 or 16..23 for the first
    // 16 rows, 8..15 or 24..31 for the others)
    static constexpr int sw_plane(int b) { return b * BM + 8 * (b & 1) + 32 * (b >> 1); }
    static constexpr size_t OFF_MW = OFF_SW + ((size_t)GEMM_KB * BM + 64) * 4;    // fp16 [BM][KB]
    static constexpr size_t OFF_MX = OFF_MW + (HAS_MIN ? (size_t)BM * GEMM_KB * 2 : 0);   // fp16 [BN][KB]
    static constexpr size_t STAGE = OFF_MX + (HAS_MIN ? (size_t)BN * GEMM_KB * 2 : 0);
    static constexpr int W_ITEMS = BM * GEMM_KB, W_PER_T = (W_ITEMS + NT - 1) / NT;
    static constexpr int B_INSTR = BN / 8;                                        // wave instructions that fill B: 8 tokens each
    static constexpr int B_PER_W = B_INSTR / NW;
    static constexpr int SX_INSTR = BN / 64;                                      // 64 tokens' scale cells each
    static constexpr int S_ITEMS = BN * GEMM_KB, S_PER_T = (S_ITEMS + NT - 1) / NT;
    static_assert(B_INSTR % NW == 0 && B_PER_W >= 1, "the activation loads divide evenly over the waves");
    static_assert(SX_INSTR >= 1 && SX_INSTR <= NW, "one scale load instruction per wave at most");
    static_assert(W_ITEMS % NT == 0, "the weight items divide evenly over the threads");
    static_assert(STAGE % 16 == 0 && GEMM_KB == 4, "stage buffers keep 16-byte alignment; four scale planes");
};

constexpr int wait_vm0() { return 0x0F70; }                                      // s_waitcnt vmcnt(0) only

// M0 carries the LDS byte address of the wave's 1 KB destination; lane i's 16 bytes land at M0 + 16 i.  Inline assembly,
// because the compiler would make every later LDS read wait for a load it sees writing LDS; the kernel waits by hand
// (vmcnt(0) in front of the stage barrier).  Nothing else in the kernel may use M0 (no dynamic register indexing).
__device__ __forceinline__ void load16_into_lds(const uint8_t *src, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_addr) : "memory");
}

// TAIL: K is an odd multiple of 64, so the last stage of a row holds two blocks instead of four.  Its other two are read from
// the blocks in front of them (in bounds) with both scales set to zero, which adds 0 * (a finite sum): a template argument,
// because the selects that zero the activation scales would sit in every stage of the K % 128 == 0 shapes too.  Before this form
// such rows ran through the dot-product GEMV, a pass per 8 tokens (Q4_0, 133 tokens, 960 and 2560 rows of 960 values: 17 passes
// of 6 - 8 us, 110 - 140 us a matrix; one launch of 8 - 12 us with this kernel; an 8-layer step 5818 -> 995 us).
// NEAR: a stage's four products are summed by themselves, and what rounding takes from the sum of the stages is kept and added at the
// end.  One chain of K / 32 additions is up to 4.5 times as far from the 64-bit sum as the lanes of a GEMV (relative 2-norm, Q4_0, chain / GEMV:
// 960 values 1.0e-7 / 6.3e-8, 14336 values 3.8e-7 / 8.4e-8); this stays at 4.9e-8 whatever the length.  It costs a tenth of the walk (us, chain
// / NEAR: Q4_0 1345 rows x 1024 values at 19 tokens 11.3 / 12.3, IQ4_NL 3538 x 960 at 41 12.7 / 13.7).  Not for the types with a minimum, whose fp16 product of minima and block sums already rounds once per stage (Q4_1 960
// values: GEMV 8.8e-8, NEAR 1.09e-7).
template <int WT, int TM, int TN, int WR, int WC, int OCC, bool GATHER, bool TAIL, bool NEAR>
__global__ __launch_bounds__(WR *WC * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void gemm_blk32_kernel(GemmMats mats, int64_t K, const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M, TileMap map, RowGather rg,
                       int slice_stages) {
    using T = Blk32<WT>;
    using C = DirectCfg<TM, TN, WR, WC, T::HAS_MIN>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC;
    const int half = lane >> 5, l32 = lane & 31;
    TileCoord tc;
    int32_t entry = 0;
    if constexpr (GATHER) {
        if (!gather_tile<C::BN>(rg, map, entry, tc.row_tile)) return;
        tc.tok_tile = 0;
    } else {
        tc = xcd_tile(blockIdx.x, map);
        if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;
    }
    const GemmMat mat = GATHER ? mats.m[0] : pick_gemm_mat(mats, tc.row_tile);
    const int64_t N = mat.N, ldy = mat.ldy;
    const size_t nb01 = mat.nb01;
    float *__restrict__ y = mat.y;
    const int64_t row_base = (int64_t)tc.row_tile * C::BM;
    size_t w_offset;
    const GatherView gv = resolve_gather<GATHER>(rg, entry, w_offset, M);
    const uint8_t *__restrict__ W = mat.W + w_offset;
    const int64_t tok_base = (int64_t)(GATHER ? gv.tok_tile : tc.tok_tile) * C::BN;
    if (tok_base >= M) return;
    static_assert(!(GATHER && TAIL), "expert rows are whole stages");
    int stage0 = 0, nstages = (int)(TAIL ? ceil_div(K, (int64_t)(32 * GEMM_KB)) : K / (32 * GEMM_KB));
    int tail_stage = nstages - 1;                                                  // TAIL: the short stage, counted from this slice's first
    if (!GATHER && slice_stages > 0) {
        stage0 = (int)blockIdx.y * slice_stages;
        nstages = min(slice_stages, nstages - stage0);
        tail_stage -= stage0;
        y += (size_t)blockIdx.y * (size_t)M * (size_t)ldy;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;

    // ---- sources of this thread's share of a stage (stage 0 of the slice; they advance by a constant per stage) ----
    const uint8_t *wsrc[C::W_PER_T];
#pragma unroll
    for (int i = 0; i < C::W_PER_T; i++) {
        const int item = tid + i * C::NT, r = item / GEMM_KB, b = item % GEMM_KB;
        wsrc[i] = W + (size_t)min(row_base + r, N - 1) * nb01 + ((size_t)stage0 * GEMM_KB + b) * T::BYTES;
    }
    // activation cells: instruction q = wave * B_PER_W + j fills tokens 8 q .. 8 q + 7, lane -> token lane / 8, slot lane % 8
    const uint8_t *bsrc[C::B_PER_W];
#pragma unroll
    for (int j = 0; j < C::B_PER_W; j++) {
        const int t = (wave * C::B_PER_W + j) * 8 + (lane >> 3);
        const int cell = (lane & 7) ^ ((t >> 1) & 7);
        bsrc[j] = ws + (size_t)gv.act_row(min(tok_base + t, M - 1)) * ws_stride + (size_t)stage0 * (32 * GEMM_KB) + 16 * cell;
    }
    const uint8_t *sxsrc = ws + (size_t)gv.act_row(min(tok_base + (wave < C::SX_INSTR ? wave : 0) * 64 + lane, M - 1)) * ws_stride +
                           q8_0_off_d(K) + (size_t)stage0 * (4 * GEMM_KB);
    const uint8_t *msrc[C::S_PER_T];                                               // block_q8_1.s of the types with a minimum
    if constexpr (T::HAS_MIN) {
#pragma unroll
        for (int i = 0; i < C::S_PER_T; i++) {
            const int item = tid + i * C::NT;
            msrc[i] = ws + (size_t)gv.act_row(min(tok_base + min(item / GEMM_KB, C::BN - 1), M - 1)) * ws_stride + q8_0_off_s(K) +
                      ((size_t)stage0 * GEMM_KB + item % GEMM_KB) * 4;
        }
    }

    typename T::Raw wq[C::W_PER_T];
    uint32_t wd[C::W_PER_T];
    float xm[C::S_PER_T];
    // TAIL: the fetched items belong to the missing blocks.  Their scales are zeroed when they are committed, a stage after the
    // fetch: a select beside the load would wait for it there, in front of the stage's products (2560 x 960 at 133 tokens, with -> without
    // such a select: Q8_0 15.7 -> 13.4 us, Q5_0 15.9 -> 14.8, Q4_1 15.3 -> 14.5, Q4_0 13.8 -> 13.2).
    bool dead = false;
    static_assert(C::NT % GEMM_KB == 0, "a thread's items all have the same block index");
    auto fetch_w = [&](int s) {
        dead = TAIL && s == tail_stage && tid % GEMM_KB >= 2;
#pragma unroll
        for (int i = 0; i < C::W_PER_T; i++) {
            const uint8_t *p = wsrc[i] + (size_t)s * (GEMM_KB * T::BYTES) - (TAIL && dead ? 2 * T::BYTES : 0);
            if constexpr (T::HAS_MIN) wd[i] = *reinterpret_cast<const uint32_t *>(p);
            else wd[i] = *reinterpret_cast<const unsigned short *>(p);
            T::fetch(wq[i], p);
        }
        if constexpr (T::HAS_MIN) {
#pragma unroll
            for (int i = 0; i < C::S_PER_T; i++)
                xm[i] = *reinterpret_cast<const float *>(msrc[i] + (size_t)s * (4 * GEMM_KB) - (TAIL && dead ? 8 : 0));
        }
    };
    auto issue_direct = [&](int s, uint32_t buf_off) {
#pragma unroll
        for (int j = 0; j < C::B_PER_W; j++)
            load16_into_lds(bsrc[j] + (size_t)s * (32 * GEMM_KB),
                            __builtin_amdgcn_readfirstlane(lds0 + buf_off + (uint32_t)C::OFF_B + (uint32_t)(wave * C::B_PER_W + j) * 1024u));
        if (wave < C::SX_INSTR)
            load16_into_lds(sxsrc + (size_t)s * (4 * GEMM_KB),
                            __builtin_amdgcn_readfirstlane(lds0 + buf_off + (uint32_t)C::OFF_SX + (uint32_t)wave * 1024u));
    };
    auto commit_w = [&](uint32_t buf_off) {
        uint8_t *base = lds + buf_off;
        u32x4 *A = reinterpret_cast<u32x4 *>(base + C::OFF_A);
        float *SW = reinterpret_cast<float *>(base + C::OFF_SW);
#pragma unroll
        for (int i = 0; i < C::W_PER_T; i++) {
            const int item = tid + i * C::NT, r = item / GEMM_KB, b = item % GEMM_KB;
            if (TAIL && dead) wd[i] = 0u;
            u32x4 lo, hi;
            T::emit(wq[i], lo, hi);
            A[(b * 2 + 0) * C::A_PLANE + r] = lo;
            A[(b * 2 + 1) * C::A_PLANE + r] = hi;
            const int i32 = r & 31;
            // the lane that owns MFMA result register v of a 32-row tile holds row 8*(v/4) + 4*half + v%4: the scale of
            // row i goes to half*16 + (i/8)*4 + i%4, so a lane reads its 16 scales as one contiguous run
            const int pos = ((i32 >> 2) & 1) * 16 + (i32 >> 3) * 4 + (i32 & 3);
            SW[C::sw_plane(b) + (r & ~31) + pos] = h2f(wd[i]);
            if constexpr (T::HAS_MIN) reinterpret_cast<unsigned short *>(base + C::OFF_MW)[r * GEMM_KB + b] = (unsigned short)(wd[i] >> 16);
        }
        if constexpr (T::HAS_MIN) {
#pragma unroll
            for (int i = 0; i < C::S_PER_T; i++) {
                const int item = tid + i * C::NT;
                if (C::S_ITEMS % C::NT == 0 || item < C::S_ITEMS)
                    reinterpret_cast<unsigned short *>(base + C::OFF_MX)[item] = f2h_rne(TAIL && dead ? 0.f : xm[i]);      // [token][KB]; exact
            }
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int c = 0; c < TN; c++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[a][c][v] = 0.f;
    float sum[NEAR ? TM : 1][NEAR ? TN : 1][16] = {}, off[NEAR ? TM : 1][NEAR ? TN : 1][16] = {};
    i32x16 magic;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        int m = MAGIC_I;
        asm volatile("" : "+v"(m));
        magic[v] = m;
    }

    // per-lane LDS byte offsets inside a stage buffer; everything else is an immediate
    const int r0 = wr * TM * 32, n0 = wc * TN * 32;
    const uint32_t a_rd = (uint32_t)C::OFF_A + (uint32_t)(half * C::A_PLANE + r0 + l32) * 16u;
    const uint32_t sw_rd = (uint32_t)C::OFF_SW + (uint32_t)(r0 + half * 16) * 4u;
    const uint32_t sx_rd = (uint32_t)C::OFF_SX + (uint32_t)(n0 + l32) * 16u;
    uint32_t b_rd[GEMM_KB];
#pragma unroll
    for (int b = 0; b < GEMM_KB; b++) b_rd[b] = (uint32_t)C::OFF_B + (uint32_t)(n0 + l32) * 128u + 16u * (uint32_t)((2 * b + half) ^ ((l32 >> 1) & 7));

    // one stage from the buffer at byte offset BUF
    auto compute = [&](auto buf_tag, int s) {
        constexpr uint32_t BUF = decltype(buf_tag)::value ? (uint32_t)C::STAGE : 0u;
        const uint8_t *base = lds + BUF;
        if constexpr (T::HAS_MIN) {
            f16x4 ma[TM], sb[TN];
#pragma unroll
            for (int a = 0; a < TM; a++) {
                const u32x2 t = reinterpret_cast<const u32x2 *>(base + C::OFF_MW)[r0 + a * 32 + l32];
                ma[a] = __builtin_bit_cast(f16x4, half ? u32x2{0u, 0u} : t);
            }
#pragma unroll
            for (int c = 0; c < TN; c++) {
                const u32x2 t = reinterpret_cast<const u32x2 *>(base + C::OFF_MX)[n0 + c * 32 + l32];
                sb[c] = __builtin_bit_cast(f16x4, half ? u32x2{0u, 0u} : t);
            }
#pragma unroll
            for (int a = 0; a < TM; a++)
#pragma unroll
                for (int c = 0; c < TN; c++) acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x8f16(ma[a], sb[c], acc[a][c], 0, 0, 0);
        }
        float dxs[TN][GEMM_KB];
#pragma unroll
        for (int c = 0; c < TN; c++) {
            const float4 t = *reinterpret_cast<const float4 *>(base + sx_rd + c * 512);
            dxs[c][0] = t.x; dxs[c][1] = t.y; dxs[c][2] = t.z; dxs[c][3] = t.w;
            // the scale cell of the short stage ends in two words of the sums plane: any bits, NaN patterns among them
            if constexpr (TAIL) { dxs[c][2] = s == tail_stage ? 0.f : dxs[c][2]; dxs[c][3] = s == tail_stage ? 0.f : dxs[c][3]; }
            if constexpr (T::HAS_MIN) {
#pragma unroll
                for (int b = 0; b < GEMM_KB; b++) dxs[c][b] *= T::INV_MULT;       // the min term has no power of two to take back
            }
        }
        // operand registers of two k-blocks: those of k-block b + 1 are requested while k-block b is worked on, and the
        // first MFMA of k-block b + 1 is issued before the last scaling group of k-block b.  The 16 weight scales of a
        // (k-block, row tile) pair - fp32 in LDS: a mixed-precision FMA that reads them as fp16 issues at a lower rate
        // than a plain one - serve the pair's TN tiles and are requested one pair ahead, in two register sets.
        i32x4 af[2][TM], bf[2][TN];
        float swf[2][16];
        auto load_operands = [&](int b, int slot) {
#pragma unroll
            for (int a = 0; a < TM; a++) {
                const u32x4 t = *reinterpret_cast<const u32x4 *>(base + a_rd + (b * 2 * C::A_PLANE + a * 32) * 16);
                af[slot][a] = i32x4{(int)t.x, (int)t.y, (int)t.z, (int)t.w};
            }
#pragma unroll
            for (int c = 0; c < TN; c++) {
                const u32x4 t = *reinterpret_cast<const u32x4 *>(base + b_rd[b] + c * 4096);
                bf[slot][c] = i32x4{(int)t.x, (int)t.y, (int)t.z, (int)t.w};
            }
        };
        auto load_scales = [&](int g) {                                       // pair g = b * TM + a
            const int b = g / TM, a = g % TM;
            const float4 *sp = reinterpret_cast<const float4 *>(base + sw_rd + (C::sw_plane(b) + a * 32) * 4);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 t = sp[q];
                swf[g & 1][4 * q] = t.x; swf[g & 1][4 * q + 1] = t.y; swf[g & 1][4 * q + 2] = t.z; swf[g & 1][4 * q + 3] = t.w;
            }
        };
        load_operands(0, 0);
        load_scales(0);
        i32x16 d_cur = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[0][0], bf[0][0], magic, 0, 0, 0);
#pragma unroll
        for (int b = 0; b < GEMM_KB; b++) {
            const int slot = b & 1;
            if (b + 1 < GEMM_KB) load_operands(b + 1, slot ^ 1);
            float dx[TN], ndx[TN];
#pragma unroll
            for (int c = 0; c < TN; c++) {
                dx[c] = dxs[c][b];
                ndx[c] = -MAGIC_F * dx[c];
            }
#pragma unroll
            for (int a = 0; a < TM; a++) {
                const int g = b * TM + a;
                if (g + 1 < GEMM_KB * TM) load_scales(g + 1);
#pragma unroll
                for (int c = 0; c < TN; c++) {
                    i32x16 d_next = d_cur;
                    if (c + 1 < TN) d_next = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[slot][a], bf[slot][c + 1], magic, 0, 0, 0);
                    else if (a + 1 < TM) d_next = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[slot][a + 1], bf[slot][0], magic, 0, 0, 0);
                    else if (b + 1 < GEMM_KB) d_next = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[slot ^ 1][0], bf[slot ^ 1][0], magic, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);                // the MFMA goes first: it runs behind the scaling below
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float t = __builtin_fmaf(__int_as_float(d_cur[v]), dx[c], ndx[c]);
                        acc[a][c][v] = __builtin_fmaf(t, swf[g & 1][v], acc[a][c][v]);
                    }
                    d_cur = d_next;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if constexpr (NEAR) {
#pragma unroll
            for (int a = 0; a < TM; a++)
#pragma unroll
                for (int c = 0; c < TN; c++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float t = sum[a][c][v] + acc[a][c][v];
                        off[a][c][v] += acc[a][c][v] - (t - sum[a][c][v]);
                        sum[a][c][v] = t;
                        acc[a][c][v] = 0.f;
                    }
        }
    };

    // Every load gets a whole stage to arrive.  A stage begins by expanding the weights fetched during the previous stage
    // into the idle buffer (the compiler's own wait for them is exact: nothing younger is outstanding then), then requests
    // the next stage's activations (into that same idle buffer) and the weights of the stage after, and only then starts
    // its arithmetic.  In front of the barrier a wave waits until at most its weight loads - the youngest requests - are
    // outstanding, i.e. for the activations; the barrier publishes them and the expanded weights.
    // Nothing inside a stage is conditional (a branch would end the scheduling region that keeps the MFMAs and their
    // scaling interleaved): stages past the last one are the last one again, loaded and expanded into the idle buffer.
    constexpr int W_LOADS = C::W_PER_T * 2 + (T::HAS_MIN ? C::S_PER_T : 0);          // vector loads of one fetch_w
    constexpr int WAIT_ACTS = 0x0F70 | (W_LOADS & 15) | ((W_LOADS >> 4) << 14);      // s_waitcnt vmcnt(W_LOADS)
    const int last = nstages - 1;
    fetch_w(0);
    issue_direct(0, 0u);
    commit_w(0u);
    fetch_w(min(1, last));
    __builtin_amdgcn_s_waitcnt(WAIT_ACTS);
    __syncthreads();
    for (int s = 0; s < nstages; s += 2) {
        {
            commit_w((uint32_t)C::STAGE);
            issue_direct(min(s + 1, last), (uint32_t)C::STAGE);
            fetch_w(min(s + 2, last));
            compute(std::false_type{}, s);
            __builtin_amdgcn_s_waitcnt(WAIT_ACTS);
            __syncthreads();
        }
        if (s + 1 < nstages) {
            commit_w(0u);
            issue_direct(min(s + 2, last), 0u);
            fetch_w(min(s + 3, last));
            compute(std::true_type{}, s + 1);
            __builtin_amdgcn_s_waitcnt(WAIT_ACTS);
            __syncthreads();
        }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm0());
    if constexpr (NEAR) {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int c = 0; c < TN; c++)
#pragma unroll
                for (int v = 0; v < 16; v++)                                        // (an infinite sum leaves NaN in off)
                    acc[a][c][v] = off[a][c][v] == off[a][c][v] ? sum[a][c][v] + off[a][c][v] : sum[a][c][v];
    }

    // ---- epilogue: register v of tile (a, c) is row 8*(v/4) + 4*half + v%4, token l32 ----
    constexpr float POST = T::HAS_MIN ? 1.f : T::INV_MULT;
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int c = 0; c < TN; c++) {
            const int64_t tok = tok_base + n0 + c * 32 + l32;
            if (tok >= M) continue;
            const int64_t orow = gv.out_row(tok);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int64_t row = row_base + r0 + a * 32 + 8 * g + 4 * half;
                float *dst = y + (size_t)orow * ldy + row;
                const float o0 = acc[a][c][4 * g] * POST, o1 = acc[a][c][4 * g + 1] * POST, o2 = acc[a][c][4 * g + 2] * POST, o3 = acc[a][c][4 * g + 3] * POST;
                if (row + 3 < N && (((uintptr_t)dst) & 15) == 0) {
                    *reinterpret_cast<float4 *>(dst) = make_float4(o0, o1, o2, o3);
                } else {
                    const float o[4] = {o0, o1, o2, o3};
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (row + e < N) dst[e] = o[e];
                }
            }
        }
}

// With few tokens the GEMM's time is its walk over K, about 0.25 us per 32-value block whatever the token count
// (33 - 37 us at K = 4096, 110 - 120 us at K = 14336), while the GEMV forms pass over the weights once per 8 or 16
// tokens at memory speed.  Up to 128 tokens on a matrix with few row tiles the walk is cut into slices
// (blk32_slices_for below: 17 - 20 us at K = 4096, 28 - 39 us at K = 14336).  The token count from which the GEMM is
// ahead, measured on 4096 x 4096, 14336 x 4096 and 4096 x 14336 (Q8_0 and Q4_0 have the matrix-core GEMV of 16 tokens
// a pass, 8 on very long rows; the other types pass once per 8 tokens or fewer):
static bool blk32_splittable(int64_t N) { return ceil_div(N, (int64_t)64) <= 384; }
// Rows too short to be split (256 to 1920 values, less than 16 stages): with the NEAR sums the walk ends before a third GEMV pass does (us,
// passes / GEMM, rows x values: Q8_0 1004 x 960 at 17 tokens 14.6 / 11.9, Q4_0 939 x 1088 at 17 16.7 / 13.5, IQ4_NL 975 x 1152 at 22 17.3 / 14.0, Q4_0
// 10594 x 960 at 31 54 / 13.8), on longer ones of them with few rows a fourth (Q5_0 949 x 1216 at 17 14.9 / 16.2; Q4_0 2222 x 1600 at 22 25.5 / 17.1)
static int64_t blk32_near_tokens(int wtype, int64_t K, int64_t N) {
    if (wtype == T_Q4_1 || wtype == T_Q5_1 || K < 256 || K > 15 * 32 * GEMM_KB) return INT64_MAX;
    return K > (wtype == T_Q5_0 ? 9 : 11) * 32 * GEMM_KB && N <= 2048 ? 25 : 17;
}
static int64_t gemm_blk32_min_tokens(int wtype, int64_t K, int64_t N, bool can_split) {
    const bool long_rows = K > 8192, big = N * K >= ((int64_t)48 << 20);
    if (can_split && blk32_splittable(N)) {
        // Rows with a short last stage, where these three types are also slower to unpack: on a small matrix a third GEMV pass over
        // one or two tokens is the cheaper (us, passes / GEMM at 17 tokens: Q4_1 320 x 2624 14.7 / 17.4, Q5_0 960 x 3648 15.8 / 18.4,
        // Q5_1 192 x 3264 at 18 tokens 15.2 / 16.2; rows beyond 4096 values 20 / 16, 2560 x 2496 22 / 17)
        if (K % (32 * GEMM_KB) != 0 && K <= 4096 && N <= 1024 && (wtype == T_Q5_0 || wtype == T_Q4_1 || wtype == T_Q5_1)) return 19;
        return (wtype == T_Q8_0 && long_rows) ? 9 : 17;
    }
    // too many row tiles to split, or no room for the partial outputs in the caller's workspace: the unsplit walk
    // (long rows with a short last stage, few of them: the walk is slower than the passes up to some 60 tokens - us, passes / GEMM,
    // 320 x 12352: Q5_0 48 tokens 67 / 97, 65 tokens 93 / 97, Q4_1 64 tokens 85 / 93, IQ4_NL 48 tokens 69 / 77, 56 tokens 78 / 77, Q8_0
    // 49 tokens 68 / 73; 320 x 8256: IQ4_NL 49 tokens 61 / 57; 2560 x 8256 at 48 tokens the GEMM is ahead)
    if (K % (32 * GEMM_KB) != 0 && long_rows && N <= 1024) return !(wtype == T_Q8_0 || wtype == T_IQ4_NL) ? 65 : K > 10240 ? 57 : 49;
    switch (wtype) {
        case T_Q8_0: return long_rows ? 49 : big ? 17 : 49;
        case T_Q4_0: return long_rows ? 65 : big ? 33 : 49;
        default:     return big ? 32 : 48;
    }
}
// few tokens that the GEMM takes by itself for its NEAR sums only
static bool blk32_near(int wtype, int64_t K, int64_t N, int64_t n) {
    return n >= blk32_near_tokens(wtype, K, N) && n < gemm_blk32_min_tokens(wtype, K, N, false);
}
bool gemm_blk32_supported(int wtype, int64_t K, int64_t N, int64_t n, bool can_split) {
    if (!(wtype == T_Q4_0 || wtype == T_Q8_0 || wtype == T_Q5_0 || wtype == T_IQ4_NL || wtype == T_Q4_1 || wtype == T_Q5_1)) return false;
    if (K < 64 || K % 64 != 0 || N < 1) return false;
    const int64_t forced = tune("CHIP_GEMM_MIN_TOKENS", 0);
    if (forced > 0) return n >= forced;
    return n >= gemm_blk32_min_tokens(wtype, K, N, can_split) || blk32_near(wtype, K, N, n);
}

// ---- split K: the partial outputs [slice][token][row] added in slice order ----
// Bound by the reads of the partial outputs.  A thread adds four consecutive rows of one token; the groups of four are counted
// per token, so that none straddles two.  With N not a multiple of 4 they lie at 4-byte alignment, and a token's last group starts
// at N - 4 and stores only the rows that the group before it has not, so that every load is a whole one.  One launch for every N: such
// an N used to take a launch per token (us of the whole product, before -> now: Q3_K 694 x 4352 at 363 tokens 909 -> 22, Q2_K 1159 x 13056
// at 69 tokens 331 -> 27, Q8_0 670 x 5312 at 1107 tokens 2403 -> 42).
// S: float, or double where K is cut into slices of one to three super-blocks (Q2_K, IQ4_XS): up to eight roundings of the whole sum would
// otherwise be most of the error (relative 2-norm, IQ4_XS 4096 values at 64 tokens 7.7e-8 with float sums, 5.8e-8 with double; the same time).
template <typename S>
__global__ __launch_bounds__(256) void sum_slices_kernel(const float *__restrict__ part, int slices, int64_t n, int64_t N,
                                                         float *__restrict__ y, int64_t ldy) {
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const int64_t groups = ceil_div(N, (int64_t)4), g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= n * groups) return;
    const int64_t t = g / groups, r = (g - t * groups) * 4, per_slice = n * N;
    if (N < 4) {                                                                     // one group of one to three rows
        for (int64_t k = 0; k < N; k++) {
            S v = 0;
            for (int s = 0; s < slices; s++) v += (S)part[(size_t)s * per_slice + t * N + k];
            y[(size_t)t * ldy + k] = (float)v;
        }
        return;
    }
    const int64_t first = r < N - 4 ? r : N - 4;
    const float *src = part + t * N + first;
    S v[4] = {0, 0, 0, 0};
    for (int s0 = 0; s0 < slices; s0 += 8) {
        f32x4_a4 p[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (s0 + j < slices) p[j] = *reinterpret_cast<const f32x4_a4 *>(src + (size_t)(s0 + j) * per_slice);
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (s0 + j < slices)
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] += (S)p[j][k];
    }
    float *dst = y + (size_t)t * ldy + first;
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (first + k >= r) dst[k] = (float)v[k];
}
hipError_t launch_sum_slices(const float *part, int slices, int64_t n, int64_t N, float *y, int64_t ldy, hipStream_t st, bool in_double) {
    if (n <= 0 || N <= 0 || slices <= 0) return hipSuccess;
    hipLaunchKernelGGL(in_double ? sum_slices_kernel<double> : sum_slices_kernel<float>, dim3((unsigned)ceil_div(n * ceil_div(N, (int64_t)4), (int64_t)256)), dim3(256), 0, st, part, slices,
                       n, N, y, ldy);
    return hipGetLastError();
}

// Slices of K for the 64 x 64 shape: about three workgroups per CU up to 128 tokens, two with more (the partial outputs
// grow with the token count), at least eight stages each.
static int blk32_slices_for(int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int forced = (int)tune("CHIP_GEMM_SLICES", 0);
    const int64_t units = ceil_div(K, (int64_t)(32 * GEMM_KB)), tiles = ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)64);
    if (forced > 0) {
        const int64_t per = ceil_div(units, (int64_t)(forced < units ? forced : units));
        return (int)ceil_div(units, per);
    }
    if (units < 16 || (M <= 128 && !blk32_splittable(N))) return 1;
    int64_t s = (M <= 128 ? 3 : 2) * cus / tiles;
    if (s > units / 8) s = units / 8;
    if (s > 16) s = 16;
    if (s < 2) return 1;
    const int64_t per = ceil_div(units, s);
    return (int)ceil_div(units, per);                                   // no empty slice
}

// Few output tiles: gemm_blk32_few_kernel, whose ks waves a workgroup share the K of a 32 x 32 tile, or the staged walk of this file, whichever
// is estimated ahead, in us of a launch.  Fitted to 707 products of 256 to 14336 values x 320 to 14336 rows at 17 to 512 tokens (11 and 19 per cent
// of spread); the walk is left where it is more than 15 per cent slower, of the types but IQ4_NL 10 where there are more tiles than CUs.  Over 934 products of
// 257 to 1024 tiles 1.22 x, one in 90 more than 3 per cent slower than the walk (IQ4_NL 4352 x 9584 at 60 tokens 1.15 x), one in 20 left to it that would be
// more than 3 per cent ahead.  us, walk / few:
// Q4_0 960 x 960 at 133 tokens 9.3 / 5.5, 2560 x 960 13.3 / 8.4, 4096 x 4096 at 17 12.1 / 9.0, at 128 20.8 / 14.5, 2048 x 2048 at 512 20.9 / 14.7; Q5_0 2048 x 2048 at 40 13.9 / 7.4; 14336 x 4096 at 32 25.0 / 25.4 and stays.
//   few    a launch; the turns of 8 waves a CU, each the fetch of a first chunk and then its chunks of 256 values, as long as a load takes or as
//          the vector work of the waves of a CU (halfway between the average and the busiest CU: by the average alone one product in 110 was more than
//          5 per cent slower than the walk, Q8_0 4352 x 4828 at 35 tokens 19.3 / 21.9)
//          Not for more tiles than the device holds workgroups of two waves, nor for more than 16 chunks a wave, where the estimate is short of what either
//          takes (us, walk / few: Q8_0 7168 x 7543 at 1042 tokens 274 / 337, Q5_0 12800 x 4687 at 778 281 / 296; Q5_1 9984 x 6009 at 89 47.5 / 56.5, IQ4_NL
//          9472 x 6334 at 82 46.2 / 53.6); nor by two waves for Q8_0 at 33 to 64 tokens where the walk, which then reads the rows once, is not cut (10 products 0.96 x,
//          768 x 11600 at 46 9.1 / 10.1)
//   walk   a launch; the turns of the workgroups a CU holds, each the fetch of a first stage and then its stages; the slice sum
// A caller without room for the slices that the walk would be cut into keeps the order of one walk over K, whatever the tile (room: the caller has it;
// a group is planned without, so that its members have the bits of their single calls).  At most 64 tiles of rows of 4096 values
// and more also split the K of the 8 waves over two workgroups (Q4_0 8192 x 320 at 64 tokens 12.0 walk, 12.6 / 10.9 in one / two; 4096 x 320 8.4 / 8.8).
struct FewPlan { int ks, slices; };              // ks 0: the walk
static float blk32_walk_us(int wtype, int64_t K, int64_t N, int64_t M, int64_t cus) {
    const int slices = blk32_slices_for(K, N, M, cus);
    const int64_t g128 = ceil_div(N, (int64_t)128) * ceil_div(M, (int64_t)128), g64x128 = ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)128);
    int64_t wgs = ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)64) * slices, per_cu = 3;
    float stage = 0.59f;                                                 // 64 x 64 tiles
    if (slices == 1 && blk32_near(wtype, K, N, M)) stage = 0.65f;
    else if (slices == 1 && 2 * g128 >= 3 * cus) { wgs = g128; per_cu = 2; stage = 2.04f; }
    else if (slices == 1 && 2 * g64x128 >= 3 * cus) { wgs = g64x128; per_cu = 2; stage = 0.95f; }
    const int64_t turns = wgs / (per_cu * cus), rest = wgs % (per_cu * cus);
    const float stages = (float)ceil_div(ceil_div(K, (int64_t)(32 * GEMM_KB)), (int64_t)slices);
    float t = 1.8f + (float)turns * (3.6f + stages * stage * (float)per_cu);
    if (rest) t += 3.6f + stages * std::max(0.59f, stage * std::max(1.f, (float)rest / (float)cus));
    return slices > 1 ? t + 2.7f + 0.9e-6f * (float)N * (float)M * (float)slices : t;
}
static FewPlan blk32_few_plan(int wtype, int64_t K, int64_t N, int64_t M, size_t nb01, int64_t cus, bool room) {
    const int64_t tiles = ceil_div(N, (int64_t)32) * ceil_div(M, (int64_t)32);
    if (K < 256 || tiles > 65536 || nb01 > ((size_t)1 << 27) || K > ((int64_t)1 << 26)) return FewPlan{0, 1};    // (rows and tokens within 32-bit reach)
    if (tiles > 4 * cus || (!room && blk32_slices_for(K, N, M, cus) > 1)) return FewPlan{0, 1};
    float best = blk32_walk_us(wtype, K, N, M, cus) / (tiles > cus && wtype != T_IQ4_NL ? 1.1f : 1.15f);
    FewPlan plan{0, 1};
    for (int ks = 2; ks <= 8; ks *= 2) {
        const int slices = ks == 8 && tiles <= 64 && K >= 4096 ? 2 : 1;
        const int64_t wgs = tiles * slices, turn = cus * (8 / ks), turns = wgs / turn, rest = wgs % turn;
        const float chunks = (float)ceil_div(2 * ceil_div(ceil_div(K / 64, (int64_t)slices), (int64_t)ks), (int64_t)8);
        if (chunks > 16 || (wtype == T_Q8_0 && ks == 2 && M > 32 && M <= 64 && blk32_slices_for(K, N, M, cus) == 1)) continue;
        float t = 2.04f + (float)turns * (1.8f + chunks * 2.62f);
        if (rest) t += 1.8f + chunks * std::max(1.72f, 0.328f * std::max((float)ks, 0.5f * ((float)(rest * ks) / (float)cus + (float)(ceil_div(rest, cus) * ks))));
        if (slices > 1) t += 3.8f + 0.9e-6f * (float)N * (float)M * (float)slices;
        if (t < best) { best = t; plan = FewPlan{ks, slices}; }
    }
    return plan;
}

template <int WT, int TM, int TN, int WR, int WC, int OCC, bool GATHER, bool NEAR = false, bool TAIL = false>
static hipError_t launch_direct(GemmMats mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim, hipStream_t st,
                                const RowGather &rg, int64_t n_as, int slices = 1, float *part = nullptr) {
    if constexpr (!GATHER && !TAIL) {
        if (K % (32 * GEMM_KB) != 0)
            return launch_direct<WT, TM, TN, WR, WC, OCC, GATHER, NEAR, true>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, slices, part);
    }
    using C = DirectCfg<TM, TN, WR, WC, Blk32<WT>::HAS_MIN>;
    const size_t lds_bytes = 2 * C::STAGE;
    if ((int64_t)lds_bytes > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_blk32_kernel<WT, TM, TN, WR, WC, OCC, GATHER, TAIL, NEAR>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, lds_bytes, lim, grant); e != hipSuccess) return e;
    const int per_cu = (int)(lds_bytes > 80 * 1024 ? 1 : (4 * OCC / C::NW > 0 ? 4 * OCC / C::NW : 1));
    const TileMap map = make_tile_map(number_row_tiles(mats, C::BM), GATHER ? 1 : ceil_div(M, C::BN), 32 * per_cu);
    const GemmMat out = mats.m[0];
    const bool split = !GATHER && slices > 1;                                     // (one matrix)
    if (split) { mats.m[0].y = part; mats.m[0].ldy = out.N; }
    const dim3 grid = GATHER ? gather_grid(map, n_as, C::NT) : dim3(map.grid, (unsigned)slices);
    hipLaunchKernelGGL(kfn, grid, dim3(C::NT), lds_bytes, st, mats, K, (const uint8_t *)ws, ws_stride, M, map, rg,
                       split ? (int)ceil_div(ceil_div(K, (int64_t)(32 * GEMM_KB)), (int64_t)slices) : 0);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return split ? launch_sum_slices(part, slices, M, out.N, out.y, out.ldy, st) : hipSuccess;
}

template <int WT>
static hipError_t launch_type(const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim, hipStream_t st,
                              const RowGather &rg, int64_t n_as, SplitK split) {
    const int64_t cus = lim.compute_units > 0 ? lim.compute_units : 256;
    if (!rg.perm) {                                                      // (the members of a group have the plan of the first)
        const GemmMat &m = mats.m[0];
        FewPlan few = blk32_few_plan(WT, K, m.N, M, m.nb01, cus, split.part != nullptr);
        if (const int f = (int)tune("CHIP_BLK32_FEW", 0); f) few = FewPlan{f % 10 == 9 ? 0 : f % 10, f / 100 + 1};
        const bool near = blk32_near(WT, K, m.N, M);
        if (few.slices > 1 && !(split.part && split.bytes >= (size_t)few.slices * (size_t)M * (size_t)m.N * sizeof(float) && (((uintptr_t)split.part) & 15) == 0))
            few.slices = 1;
        if (few.ks > 0) return launch_gemm_blk32_few(WT, few.ks, near, mats, K, ws, ws_stride, M, lim, st, few.slices, split.part);
    }
    if (!rg.perm && split.part) {
        const int64_t N = mats.m[0].N;
        const int slices = blk32_slices_for(K, N, M, cus);
        if (slices > 1 && split.bytes >= (size_t)slices * (size_t)M * (size_t)N * sizeof(float) && (((uintptr_t)split.part) & 15) == 0) {
            return launch_direct<WT, 1, 1, 2, 2, 3, false>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, slices, split.part);
        }
    }
    // What would be GEMV passes but for the NEAR sums.  Three waves a SIMD for expert groups, whose tiles are often more than 512 (iq4_nl, 16
    // pairs over 10672 rows of 512 values 43 -> 38 us), two for the few tiles of a plain product (no spills: 5 - 10 per cent ahead).
    if constexpr (!Blk32<WT>::HAS_MIN) {
        if (rg.perm && M < MOE_FEW_PAIRS) return launch_direct<WT, 1, 1, 2, 2, 3, true, true>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);
        if (!rg.perm && blk32_near(WT, K, mats.m[0].N, M)) return launch_direct<WT, 1, 1, 2, 2, 2, false, true>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);
    }
    if (rg.perm) return launch_direct<WT, 1, 1, 2, 2, 3, true>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);      // expert groups: 64 x 64 tiles
    // Two 4-wave workgroups of 128 x 128 per CU when that fills the device, else 64 x 128, else 64 x 64 (three workgroups
    // per CU).  Measured on Q4_0 with K = 4096 (us; 128 x 128 / 64 x 128 / 64 x 64 / 128 x 256 with 8 waves): 14336 x 2048
    // tokens 375 / 413 / 468 / 415, 4096 x 2048 106 / 115 / 130 / 106, 14336 x 512 103 / 110 / 114 / 102, 4096 x 512
    // 63 / 38 / 38 / 81.
    int64_t rows128 = 0, rows64 = 0;
    for (int i = 0; i < mats.count; i++) { rows128 += ceil_div(mats.m[i].N, 128); rows64 += ceil_div(mats.m[i].N, 64); }
    const int64_t g128 = rows128 * ceil_div(M, 128), g64x128 = rows64 * ceil_div(M, 128);
    const int cfg = (int)tune("CHIP_GEMM_CFG", 2 * g128 >= 3 * cus ? 3 : 2 * g64x128 >= 3 * cus ? 6 : 4);
    switch (cfg) {
        case 3: return launch_direct<WT, 2, 2, 2, 2, 2, false>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);   // 128 x 128, 4 waves
        case 4: return launch_direct<WT, 1, 1, 2, 2, 3, false>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);   // 64 x 64, 4 waves
        case 6: return launch_direct<WT, 1, 2, 2, 2, 2, false>(mats, K, ws, ws_stride, M, lim, st, rg, n_as);   // 64 x 128, 4 waves
        default: return hipErrorInvalidValue;
    }
}

int gemm_blk32_slices(int wtype, int64_t K, int64_t N, int64_t n, int compute_units) {
    if (!gemm_blk32_supported(wtype, K, N, n, true)) return 1;
    return blk32_slices_for(K, N, n, compute_units > 0 ? compute_units : 256);
}

int gemm_blk32_moe_tile_tokens() { return DirectCfg<1, 1, 2, 2, false>::BN; }   // the 64 x 64 shape serves the expert groups

static hipError_t launch_blk32_mats(int wtype, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M,
                                    const DeviceLimits &lim, hipStream_t st, const RowGather &rg, int64_t n_as, SplitK split) {
    switch (wtype) {
        case T_Q4_0:   return launch_type<T_Q4_0>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        case T_Q8_0:   return launch_type<T_Q8_0>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        case T_Q5_0:   return launch_type<T_Q5_0>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        case T_IQ4_NL: return launch_type<T_IQ4_NL>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        case T_Q4_1:   return launch_type<T_Q4_1>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        case T_Q5_1:   return launch_type<T_Q5_1>(mats, K, ws, ws_stride, M, lim, st, rg, n_as, split);
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_gemm_blk32(int wtype, const void *W, size_t nb01, int64_t K, int64_t N, const void *ws, size_t ws_stride,
                             int64_t M, float *y, int64_t ldy, const DeviceLimits &lim, hipStream_t st, const RowGather *rgp,
                             int64_t n_as, SplitK split) {
    if (M <= 0 || N <= 0 || n_as <= 0) return hipSuccess;
    return launch_blk32_mats(wtype, one_gemm_mat(W, nb01, N, y, ldy), K, ws, ws_stride, M, lim, st,
                             rgp ? *rgp : RowGather{nullptr, nullptr, nullptr, 1, 1, 0}, n_as, split);
}

// Members that run unsplit by themselves: the same bits, fewer launches (us, Q4_0 at 133 tokens x 960 values: wq + wk + wv of 960 + 320 +
// 320 rows 31 -> 13, ffn_gate + ffn_up of 2560 rows 23 -> 14; 512 tokens x 4096 values x 14336 rows twice 195 -> 185).
bool gemm_blk32_group_applicable(int wtype, int64_t K, const GemmMats &mats, int64_t n, int compute_units) {
    if (mats.count < 2) return false;
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    const FewPlan first = blk32_few_plan(wtype, K, mats.m[0].N, n, mats.m[0].nb01, cus, false);
    for (int i = 0; i < mats.count; i++) {
        const FewPlan few = blk32_few_plan(wtype, K, mats.m[i].N, n, mats.m[i].nb01, cus, false);
        if (few.ks != first.ks || few.slices != 1 || (few.ks == 0 && gemm_blk32_slices(wtype, K, mats.m[i].N, n, compute_units) != 1) ||
            !gemm_blk32_supported(wtype, K, mats.m[i].N, n, false) || blk32_near(wtype, K, mats.m[i].N, n) != blk32_near(wtype, K, mats.m[0].N, n))
            return false;
    }
    return true;
}
hipError_t launch_gemm_blk32_group(int wtype, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t n, const DeviceLimits &lim,
                                   hipStream_t st) {
    return launch_blk32_mats(wtype, mats, K, ws, ws_stride, n, lim, st, RowGather{nullptr, nullptr, nullptr, 1, 1, 0}, 1, SplitK{nullptr, 0});
}

}  // namespace chip
