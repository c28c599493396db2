// Grouping of the (token, slot) pairs of LM_GGML_OP_MUL_MAT_ID by expert, on the device: what the reference builds
// in matrix_row_counts / matrix_rows (ggml-cpu/ggml-cpu.c:1625-1640) as a counting sort, so that each expert's pairs
// can run through a GEMM over that expert's matrix.  The order of the pairs inside an expert's list is not fixed
// (atomic cursors); no output depends on it, since every output row is computed on its own.
#include "dev_common.h"
#include "kernels.h"

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

}  // namespace chip
