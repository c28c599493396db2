// Grouping of the (token, slot) pairs of LM_GGML_OP_MUL_MAT_ID by expert, on the device: what the reference builds
// in matrix_row_counts / matrix_rows (ggml-cpu/ggml-cpu.c:1625-1640) as a counting sort, so that each expert's pairs
// can run through a GEMM over that expert's matrix.  The order of the pairs inside an expert's list is not fixed
// (atomic cursors); no output depends on it, since every output row is computed on its own.
#include "dev_common.h"
#include "kernels.h"
#include <algorithm>
#include <cmath>

namespace chip {

constexpr int MOE_GROUP_THREADS = 1024;
constexpr int MOE_MAX_EXPERTS = 1 << MOE_EXPERT_BITS;   // LDS: an int32 per expert; tile entries keep 12 bits for it

// Sums of v over the lanes in front of this one; two sums side by side in one int2
__device__ __forceinline__ int2 lanes_before(int2 v) {
    const int lane = threadIdx.x & 63;
    int2 inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int a = __shfl_up(inc.x, d), b = __shfl_up(inc.y, d);
        if (lane >= d) { inc.x += a; inc.y += b; }
    }
    return make_int2(inc.x - v.x, inc.y - v.y);
}

// offsets[e] .. offsets[e+1]: expert e's stretch of perm; perm holds pair numbers token * n_used + slot.  Pairs whose
// id lies outside [0, n_as) are left out (the reference asserts on them).  tiles: the list of (expert, token tile)
// work items for tiles of tile_tokens pairs, its length in front.
// Bound: latency.  One workgroup, since everything meets in one set of counters: a load of the ids (kept in registers for the scatter,
// up to MOE_KEEP pairs a thread), LDS atomics, a scan by the first wave (four experts a lane and turn), the scatter.  512 tokens x 8 of 128
// experts 12.4 -> 6 us; before, one thread ran over the experts and the pair numbers were divided in 64 bits.
constexpr int MOE_KEEP = 8;
__global__ __launch_bounds__(MOE_GROUP_THREADS) void moe_group_kernel(const int32_t *__restrict__ ids, int64_t ids_stride,
                                                                       unsigned n_used, unsigned pairs, int n_as, int tile_tokens,
                                                                       int32_t *__restrict__ offsets, int32_t *__restrict__ perm,
                                                                       int32_t *__restrict__ tiles) {
    constexpr int PER = 4;                                          // experts of a lane in a turn of the scan
    __shared__ int32_t count[MOE_MAX_EXPERTS];
    const unsigned tid = threadIdx.x;
    auto expert = [&](unsigned p) {
        const int32_t e = ids[(int64_t)(p / n_used) * ids_stride + p % n_used];
        return (unsigned)e < (unsigned)n_as ? e : -1;
    };
    int32_t kept[MOE_KEEP];
#pragma unroll
    for (int i = 0; i < MOE_KEEP; i++) {
        kept[i] = -1;
        if (i * MOE_GROUP_THREADS >= pairs) continue;                // the same for all threads
        const unsigned p = tid + i * MOE_GROUP_THREADS;
        if (p < pairs) kept[i] = expert(p);
    }
    for (int e = tid; e < n_as; e += MOE_GROUP_THREADS) count[e] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MOE_KEEP; i++)
        if (kept[i] >= 0) atomicAdd(&count[kept[i]], 1);
    for (unsigned p = tid + MOE_KEEP * MOE_GROUP_THREADS; p < pairs; p += MOE_GROUP_THREADS) {
        const int32_t e = expert(p);
        if (e >= 0) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (tid < 64) {
        int2 base = make_int2(0, 0);                                 // pairs and tiles of the experts of earlier turns
        for (int e0 = 0; e0 < n_as; e0 += 64 * PER) {
            int c[PER];
            int2 mine = make_int2(0, 0);
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int e = e0 + (int)tid * PER + i;
                c[i] = e < n_as ? count[e] : 0;
                mine.x += c[i];
                mine.y += (c[i] + tile_tokens - 1) / tile_tokens;
            }
            int2 at = lanes_before(mine);
            at.x += base.x;
            at.y += base.y;
            base = make_int2(__shfl(at.x + mine.x, 63), __shfl(at.y + mine.y, 63));
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int e = e0 + (int)tid * PER + i;
                if (e >= n_as) break;
                offsets[e] = at.x;
                count[e] = at.x;                                     // from here on the write cursor
                const int nt = (c[i] + tile_tokens - 1) / tile_tokens;
                for (int t = 0; t < nt; t++) tiles[1 + at.y + t] = e | (t << MOE_EXPERT_BITS);
                at.x += c[i];
                at.y += nt;
            }
        }
        if (tid == 0) { tiles[0] = base.y; offsets[n_as] = base.x; }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MOE_KEEP; i++)
        if (kept[i] >= 0) perm[atomicAdd(&count[kept[i]], 1)] = (int32_t)(tid + i * MOE_GROUP_THREADS);
    for (unsigned p = tid + MOE_KEEP * MOE_GROUP_THREADS; p < pairs; p += MOE_GROUP_THREADS) {
        const int32_t e = expert(p);
        if (e >= 0) perm[atomicAdd(&count[e], 1)] = (int32_t)p;
    }
}

bool moe_group_supported(int64_t n_as, int64_t pairs) {
    return n_as >= 1 && n_as <= MOE_MAX_EXPERTS && pairs / 64 + n_as < ((int64_t)1 << (31 - MOE_EXPERT_BITS)) && pairs / 64 + n_as <= 65535;
}

hipError_t launch_moe_group(const int32_t *ids, int64_t ids_stride, int64_t n_used, int64_t pairs, int64_t n_as,
                            int tile_tokens, int32_t *offsets, int32_t *perm, int32_t *tiles, hipStream_t st) {
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(MOE_GROUP_THREADS), 0, st, ids, ids_stride, (unsigned)n_used, (unsigned)pairs, (int)n_as,
                       tile_tokens, offsets, perm, tiles);
    return hipGetLastError();
}

// Few pairs of long rows stay with the GEMV, whose lanes share the additions that the GEMM makes in one chain of K / 256 (error, relative 2-norm
// x 1e8, GEMV / GEMM: Q4_K 4096 values 12.7 / 10.2, 8192 12.6 / 12.2, 14336 12.8 / 15.1; Q6_K 2048 7.2 / 5.9, 4096 7.7 / 8.0, 14336 8.3 / 13.2;
// Q2_K 4096 11.0 / 8.6, 8192 10.7 / 11.5; Q5_K as Q4_K, Q3_K and IQ4_XS as Q6_K).  The types with a minimum per 32 values as well, at every length;
// the other block-32 types have sums of their own for this.
static bool few_pairs_as_near(int wtype, int64_t K) {
    switch (wtype) {
        case T_Q4_1: case T_Q5_1: return false;
        case T_Q4_K: case T_Q5_K: return K <= 8192;
        case T_Q2_K: return K <= 4096;
        case T_Q6_K: case T_Q3_K: case T_IQ4_XS: return K < 4096;
        default: return true;
    }
}

// MUL_MAT_ID: the pairs grouped by expert and run through the GEMM of the weight type, or a GEMV per pair?  Both times estimated in us, with
// terms fitted to 40 measured products of each type and checked against 14500 others (16 to 4095 pairs, 2 to 400 experts, 256 to 14336 values, at most 1 GB
// of experts that no cache holds):
//   GEMV   a pair costs its rows by the 4096 values of one of them; that pairs share an expert buys nothing.  From 64 pairs on not faster than
//          8 TB/s, which large experts come to (Q8_0 3072 values x 1024 rows, 32 experts, 156 pairs 69, 42 without this term; GEMM 38); fewer
//          pairs share the caches (Q8_0 2048 x 3584, 8 experts, 32 pairs 29, 38 with it)
//   GEMM   quantizer, grouping and launch, a walk over K, and the tiles by the 512 that the chip runs at a time.  With ids drawn evenly
//          n_as * (1 - e^(-pairs / n_as)) experts are picked, and a single pair has its row tiles walked whole
// Where both are close the choice is the one on the safer side of the estimates (nine in ten within 20 per cent, the worst 40 to 80): the GEMV below 64
// pairs and for Q2_K, Q3_K and IQ4_XS, else the GEMM.
// (us, GEMV / GEMM: Q4_K 2048 values x 768 rows, 128 experts, 64 pairs 17 / 26, 128 pairs 28.5 / 28.2; 768 x 2048 64 pairs 34 / 24; 4096 x
// 14336, 8 experts, 16 pairs 63 / 70, 32 pairs 105 / 69; Q4_0 2560 x 12214, 12 experts, 32 pairs 71 / 96; Q8_0 1024 x 3676, 28 experts, 32 pairs
// 30 / 45.  Of the 14500 calls 3 per cent take the slower one by more than 5 per cent, and 7 calls by 5 to 15 per cent where the line at 64 pairs
// takes the faster; that line takes the slower one by more than 5 per cent in 15 per cent of them.)  F16 stays with the line: its GEMV's time is that of the experts' bytes.
bool moe_gemm_ahead(int wtype, int64_t K, int64_t N, size_t row_bytes, int64_t n_as, int64_t pairs) {
    const int64_t forced = tune("CHIP_MOE_MIN", 0);
    if (forced > 0) return pairs >= forced;
    if (wtype == T_F16 || gemv_max_tokens(wtype, K, DeviceLimits{256, 160 * 1024}) < 1) return pairs >= MOE_FEW_PAIRS;
    if (pairs < 16 || pairs >= 4096) return pairs >= 16;
    const bool few = pairs < MOE_FEW_PAIRS;
    if (few && !few_pairs_as_near(wtype, K)) return false;
    struct { float pair, walk, turn, ends; } c;                         // pair: per 1024 rows x 4096 values; the others per super-block, per tile
    const bool low_bit = wtype == T_Q3_K || wtype == T_Q2_K || wtype == T_IQ4_XS;
    switch (wtype) {
        case T_Q4_K:   c = {0.235f, 0.92f, 1.25f, 3.5f}; break;
        case T_Q5_K:   c = {0.365f, 1.10f, 1.50f, 4.0f}; break;
        case T_Q6_K:   c = {0.390f, 1.50f, 1.55f, 5.0f}; break;
        case T_Q3_K:   c = {0.355f, 0.90f, 1.30f, 3.5f}; break;
        case T_Q2_K:   c = {0.255f, 0.80f, 1.20f, 3.5f}; break;
        case T_IQ4_XS: c = {0.390f, 1.30f, 1.80f, 3.5f}; break;
        case T_Q8_0:   c = {0.230f, 1.00f, 1.60f, 2.0f}; break;
        case T_Q4_0:   c = {0.170f, 1.00f, 0.95f, 2.2f}; break;
        case T_Q5_0:   c = {0.300f, 1.60f, 1.00f, 3.0f}; break;
        case T_Q4_1:   c = {0.200f, 1.30f, 1.00f, 2.0f}; break;
        case T_Q5_1:   c = {0.300f, 1.45f, 1.00f, 2.4f}; break;
        default:       c = {0.380f, 1.07f, 1.05f, 2.1f};                // IQ4_NL
    }
    const float n_pairs = (float)pairs, experts = (float)n_as, units = (float)K / 256.f;
    const float pair_bytes = (float)N * (float)row_bytes;
    const float gemv = 6.5f + n_pairs * std::max(c.pair * (float)N / 1024.f * (float)ceil_div(K, (int64_t)4096), few ? 0.f : pair_bytes / 8e6f);
    const float tiles = (experts * (1.f - std::exp(-n_pairs / experts)) + n_pairs / 64.f) * (float)ceil_div(N, (int64_t)(gemm_kq_type(wtype) ? 128 : 64));
    const float gemm = 10.f + c.walk * units + tiles / 512.f * (c.turn * units + c.ends);
    return gemm * (few ? 1.15f : low_bit ? 1.05f : 0.95f) < gemv;
}

}  // namespace chip
