// GEMM for gfx950 over weights in 32-value blocks (Q4_0, Q8_0, Q5_0, IQ4_NL; Q4_1 and Q5_1 with a minimum on top) for products with few output
// tiles: the batched form of lm_ggml_vec_dot_q4_0_q8_0 .. _iq4_nl_q8_0 (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449), Y[t][r] = sum_b dw[r][b] * dx[t][b] * isum[t][r][b].
//
// gemm_blk32_kernel walks K in stages that wait for each other: with fewer tiles than the device holds workgroups a product takes as long as
// one walk, most of a microsecond a stage, and cutting K over the grid costs a second launch.  Here the waves of a workgroup share one tile of
// 32 rows x 32 tokens and cut K between them, and each is on its own until the end: it loads its rows' packed bytes and its tokens' quants in
// memory order, a chunk of eight blocks ahead of the one it multiplies, and turns them round through a stretch of LDS of its own, with no
// barrier.  The waves' sums meet in LDS once and are added in order.
//
// Both scales of a block come from fp16, so their products over a tile are one v_mfma_f32_32x32x8f16 with one live k (22-bit significands,
// exact in fp32): no scale is read per result, and a result is out += (bits(12582912 + isum) - 12582912) * (dw * dx).  The four blocks of half a
// chunk are summed by themselves and what rounding takes from the sum of the halves is kept (NEAR, for the calls that ran so before), or a
// chunk's eight are, and the chunks' sums are added; the waves' in 64 bits.  Relative 2-norm of the error against 64-bit sums, walk / this / NEAR:
// Q4_0 960 values 1.0e-7 / 5.9e-8 / 4.9e-8, 14336 values 1.3e-7 / 8.0e-8 / 4.9e-8.
//
// Bound: the issue of vector instructions, by the counters some 450 per chunk and wave (two per result, the unpacking, the sums) and 350 a wave to start and
// to add up, at two waves a SIMD: 2.1 us a chunk of 8 waves on a CU (Q4_0 4096 rows at 64 tokens 17.2 us for 8192 values, 21.4 for 12288).  Registers (210 to
// 250) hold a third wave off.  Loading operands straight from
// global memory, a lane its own row's, took twice as long: 32 rows a load instruction cost some 160 clocks of the CU's address unit.  us,
// gemm_blk32_kernel / this, values x rows: Q4_0 960 x 960 at 133 tokens 9.3 / 5.5, 4096 x 4096 at 17 12.1 / 9.0, 2048 x 2048 at 512 20.9 / 14.7.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include <type_traits>

namespace chip {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int CHUNK = 8;                      // 32-value blocks a wave loads at a time
constexpr float MAGIC_F = 12582912.f;         // 1.5 * 2^23: an MFMA whose C input holds its bits leaves bits(12582912 + isum), |isum| < 2^22
constexpr int MAGIC_I = 0x4B400000;

__device__ __forceinline__ uint32_t spread4(uint32_t bits) { return ((bits & 0xfu) * 0x00204081u) & 0x01010101u; }   // bit k -> bit 8k
__device__ __forceinline__ uint32_t iq4_lookup(uint32_t idx) {                // four indices -> code points of kvalues_iq4nl
    constexpr uint32_t T0 = 0xbfad9881u, T1 = 0xf6eaddcfu, T2 = 0x26190d01u, T3 = 0x71594535u;
    const uint32_t sel = idx & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
    return __builtin_amdgcn_perm(hi, lo, ((idx >> 1) & 0x04040404u) | 0x03020100u);
}

// Per type: two neighbouring blocks (4-byte aligned whatever the type), of which a lane reads D dwords from byte `at(half)` on, and what it makes
// of them: the 16 signed bytes of its k-half of either block times 1 / POST, and the words whose low (first block) and high half (second)
// hold d, and the minimum.  A lane of k-half 1 needs no scale.
struct Pair { u32x4 c0, c1; uint32_t d0, d1, m; };
template <int WT> struct Few;
template <> struct Few<T_Q4_0> {
    static constexpr int BYTES = BYTES_Q4_0, D = 9;
    static constexpr bool HAS_MIN = false;
    static constexpr float POST = 1.f / 16.f;
    __device__ static __forceinline__ int at(int) { return 0; }
    __device__ static __forceinline__ uint32_t cell(uint32_t q, int half) { return ((q << (4 - 4 * half)) & 0xf0f0f0f0u) ^ 0x80808080u; }   // 16 * (nibble - 8)
    template <typename F> __device__ static __forceinline__ Pair nibbles(const uint32_t (&w)[D], F cell) {
        Pair p;
#pragma unroll
        for (int i = 0; i < 4; i++) { p.c0[i] = cell(shr16(w[i + 1], w[i])); p.c1[i] = cell(w[5 + i]); }
        p.d0 = w[0]; p.d1 = w[4]; p.m = 0u;
        return p;
    }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int half) {
        return nibbles(w, [half](uint32_t q) { return cell(q, half); });
    }
};
template <> struct Few<T_IQ4_NL> {
    static constexpr int BYTES = BYTES_IQ4_NL, D = 9;
    static constexpr bool HAS_MIN = false;
    static constexpr float POST = 1.f;
    __device__ static __forceinline__ int at(int) { return 0; }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int half) {
        return Few<T_Q4_0>::nibbles(w, [half](uint32_t q) { return iq4_lookup((q >> (4 * half)) & 0x0f0f0f0fu); });
    }
};
template <> struct Few<T_Q8_0> {
    static constexpr int BYTES = BYTES_Q8_0, D = 10;                 // dwords 4 half .. 4 half + 4 and 8 + 4 half .. 12 + 4 half of the 17
    static constexpr bool HAS_MIN = false;
    static constexpr float POST = 1.f;
    __device__ static __forceinline__ int at(int half) { return 16 * half; }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int) {
        Pair p;
#pragma unroll
        for (int i = 0; i < 4; i++) { p.c0[i] = shr16(w[i + 1], w[i]); p.c1[i] = w[6 + i]; }
        p.d0 = w[0]; p.d1 = w[5]; p.m = 0u;
        return p;
    }
};
template <> struct Few<T_Q5_0> {
    static constexpr int BYTES = BYTES_Q5_0, D = 11;
    static constexpr bool HAS_MIN = false;
    static constexpr float POST = 1.f / 8.f;
    __device__ static __forceinline__ int at(int) { return 0; }
    // 8 * (q - 16): element j of a k-half has bit j of its half of qh on top
    __device__ static __forceinline__ uint32_t cell(uint32_t q, uint32_t hb, int i, int half) {
        return ((((q >> (4 * half)) & 0x0f0f0f0fu) << 3) | (spread4(hb >> (4 * i)) << 7)) ^ 0x80808080u;
    }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int half) {
        Pair p;
        const uint32_t h0 = shr16(w[1], w[0]) >> (16 * half), h1 = w[6] >> (16 * half);
#pragma unroll
        for (int i = 0; i < 4; i++) { p.c0[i] = cell(shr16(w[i + 2], w[i + 1]), h0, i, half); p.c1[i] = cell(w[7 + i], h1, i, half); }
        p.d0 = w[0]; p.d1 = w[5]; p.m = 0u;
        return p;
    }
};
template <> struct Few<T_Q4_1> {
    static constexpr int BYTES = BYTES_Q4_1, D = 10;
    static constexpr bool HAS_MIN = true;
    static constexpr float POST = 1.f;
    __device__ static __forceinline__ int at(int) { return 0; }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int half) {
        Pair p;
#pragma unroll
        for (int i = 0; i < 4; i++) { p.c0[i] = (w[1 + i] >> (4 * half)) & 0x0f0f0f0fu; p.c1[i] = (w[6 + i] >> (4 * half)) & 0x0f0f0f0fu; }
        p.d0 = w[0]; p.d1 = w[5] << 16; p.m = (w[0] >> 16) | (w[5] & 0xffff0000u);
        return p;
    }
};
template <> struct Few<T_Q5_1> {
    static constexpr int BYTES = BYTES_Q5_1, D = 12;
    static constexpr bool HAS_MIN = true;
    static constexpr float POST = 1.f;
    __device__ static __forceinline__ int at(int) { return 0; }
    __device__ static __forceinline__ Pair pair(const uint32_t (&w)[D], int half) {
        Pair p;
        const uint32_t h0 = w[1] >> (16 * half), h1 = w[7] >> (16 * half);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p.c0[i] = ((w[2 + i] >> (4 * half)) & 0x0f0f0f0fu) | (spread4(h0 >> (4 * i)) << 4);
            p.c1[i] = ((w[8 + i] >> (4 * half)) & 0x0f0f0f0fu) | (spread4(h1 >> (4 * i)) << 4);
        }
        p.d0 = w[0]; p.d1 = w[6] << 16; p.m = (w[0] >> 16) | (w[6] & 0xffff0000u);
        return p;
    }
};

template <int WT, int KS>
struct FewCfg {
    using T = Few<WT>;
    static constexpr int NCH = CHUNK * T::BYTES / 16;                 // 16-byte pieces of a row and chunk
    static constexpr int NLD = (32 * NCH + 63) / 64;                  // loads of a lane
    // a wave's stretch: the rows of a chunk, the tokens' quants ([token][16 cells], swizzled), their scales and sums as fp16 ([token][8])
    static constexpr int OFF_X = NLD * 1024, OFF_D = OFF_X + 32 * 256, OFF_S = OFF_D + 32 * 16, WAVE = OFF_S + (T::HAS_MIN ? 32 * 16 : 0);
    static constexpr size_t LDS = (size_t)KS * WAVE;
    static_assert(CHUNK * T::BYTES % 16 == 0 && WAVE >= 8192 && WAVE % 16 == 0, "whole pieces; a wave's sums take the place of its operands");
};

template <int WT, int KS, bool NEAR>
__global__ __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_blk32_few_kernel(GemmMats mats, int64_t K, const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M, TileMap map, int slice_pairs) {
    using T = Few<WT>;
    using C = FewCfg<WT, KS>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    TileCoord tc = xcd_tile(blockIdx.x, map);
    if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;            // padding of the tile map
    const GemmMat mat = pick_gemm_mat(mats, tc.row_tile);
    const int64_t N = mat.N, row_base = (int64_t)tc.row_tile * 32, tok_base = (int64_t)tc.tok_tile * 32;
    const int tokens = (int)min((int64_t)32, M - tok_base);
    uint8_t *const own = lds + (size_t)wave * C::WAVE;

    // this wave's blocks: pairs of blocks, dealt out evenly
    const int nb = (int)(K / 32);
    int pair0 = 0, pairs = nb / 2;
    if (slice_pairs > 0) {
        pair0 = (int)blockIdx.y * slice_pairs;
        pairs = min(slice_pairs, pairs - pair0);
    }
    const int b0 = 2 * (pair0 + pairs * wave / KS), b1 = 2 * (pair0 + pairs * (wave + 1) / KS);

    // (offsets of 32 bits from the tile's first row and first token: launch_gemm_blk32_few)
    const uint8_t *const w0 = mat.W + (size_t)min(row_base, N - 1) * mat.nb01, *const x0 = ws + (size_t)tok_base * ws_stride;
    uint32_t woff[C::NLD], xoff[8];
#pragma unroll
    for (int t = 0; t < C::NLD; t++) {
        const int i = min(lane + 64 * t, 32 * C::NCH - 1), r = i / C::NCH, c = i % C::NCH;
        woff[t] = (uint32_t)(min(row_base + r, N - 1) - min(row_base, N - 1)) * (uint32_t)mat.nb01 + 16u * c;
    }
#pragma unroll
    for (int t = 0; t < 8; t++) xoff[t] = (uint32_t)min(4 * t + (lane >> 4), tokens - 1) * (uint32_t)ws_stride + 16u * (lane & 15);
    const uint32_t soff = (uint32_t)min(lane >> 1, tokens - 1) * (uint32_t)ws_stride + 16u * (lane & 1);

    struct Chunk {
        u32x4 w[C::NLD], x[8], d, s;
    };
    // the eight blocks from `at` on, which all lie in the row
    auto load = [&](Chunk &k, int at) {
#pragma unroll
        for (int t = 0; t < C::NLD; t++) k.w[t] = *reinterpret_cast<const u32x4_a4 *>(w0 + (size_t)at * T::BYTES + woff[t]);
#pragma unroll
        for (int t = 0; t < 8; t++) k.x[t] = *reinterpret_cast<const u32x4 *>(x0 + 32 * at + xoff[t]);
        k.d = *reinterpret_cast<const u32x4_a4 *>(x0 + q8_0_off_d(K) + 4 * at + soff);
        if constexpr (T::HAS_MIN) k.s = *reinterpret_cast<const u32x4_a4 *>(x0 + q8_0_off_s(K) + 4 * at + soff);
    };
    auto halves = [](const u32x4 &v) {                                                   // exact: these floats come from fp16
        return u32x2{(uint32_t)f2h_rne(__uint_as_float(v.x)) | (uint32_t)f2h_rne(__uint_as_float(v.y)) << 16,
                     (uint32_t)f2h_rne(__uint_as_float(v.z)) | (uint32_t)f2h_rne(__uint_as_float(v.w)) << 16};
    };
    auto commit = [&](const Chunk &k) {
#pragma unroll
        for (int t = 0; t < C::NLD; t++) reinterpret_cast<u32x4 *>(own)[lane + 64 * t] = k.w[t];
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int tok = 4 * t + (lane >> 4);
            reinterpret_cast<u32x4 *>(own + C::OFF_X)[tok * 16 + ((lane & 15) ^ (tok & 15))] = k.x[t];
        }
        reinterpret_cast<u32x2 *>(own + C::OFF_D)[lane] = halves(k.d);
        if constexpr (T::HAS_MIN) reinterpret_cast<u32x2 *>(own + C::OFF_S)[lane] = halves(k.s);
    };

    constexpr bool MAGIC = !(NEAR && (T::HAS_MIN || WT == T_Q8_0));                      // these have no registers left for it
    i32x16 magic;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        int m = MAGIC ? MAGIC_I : 0;
        if constexpr (MAGIC) asm volatile("" : "+v"(m));
        magic[v] = m;
    }
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const uint32_t first = half ? 0u : 0x0000ffffu, second = half ? 0u : 0xffff0000u;    // where a pair's two scales stand in k
    auto isum = [](int d) { return MAGIC ? __int_as_float(d) - MAGIC_F : (float)d; };
    float sum[16] = {}, off[NEAR ? 16 : 1] = {};
    auto scales = [&](uint32_t dx, uint32_t dw) {
        return __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(f16x4, u32x2{dx, 0u}), __builtin_bit_cast(f16x4, u32x2{dw, 0u}), zero, 0, 0, 0);
    };
    // blocks 4h .. 4h + 3 of the chunk in LDS, of which [lo, hi) count
    auto multiply = [&](auto h_tag, int lo, int hi, f32x16 &acc) {
        constexpr int H = decltype(h_tag)::value;
        const u32x4 dx4 = reinterpret_cast<const u32x4 *>(own + C::OFF_D)[l32];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint8_t *src = own + l32 * (16 * C::NCH) + (2 * H + p) * 2 * T::BYTES + T::at(half);
            uint32_t w[T::D];
#pragma unroll
            for (int i = 0; i < T::D; i++) w[i] = reinterpret_cast<const uint32_t *>(src)[WT == T_Q8_0 && i >= 5 ? i + 3 : i];
            u32x4 a[2];
#pragma unroll
            for (int j = 0; j < 2; j++) a[j] = reinterpret_cast<const u32x4 *>(own + C::OFF_X)[l32 * 16 + ((2 * (4 * H + 2 * p + j) + half) ^ (l32 & 15))];
            Pair q = T::pair(w, half);
            // a pair's products behind the sums of the one before: all at once they do not fit the registers
            if (p > 0) asm volatile("" : "+v"(acc), "+v"(q.c0), "+v"(q.c1));
            const uint32_t live = 4 * H + 2 * p >= lo && 4 * H + 2 * p < hi ? 0xffffffffu : 0u;       // (lo and hi are even)
            const uint32_t dx = dx4[2 * H + p] & live;                                  // (both factors: a block that does not count may have an infinite one)
            const i32x16 D0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a[0]), __builtin_bit_cast(i32x4, q.c0), magic, 0, 0, 0);
            const f32x16 P0 = scales(dx & first, q.d0 & first & live);
            if constexpr (T::HAS_MIN) {                                             // m[r][b] * s[t][b]: fp16 factors on both sides
                const uint32_t s = reinterpret_cast<const u32x4 *>(own + C::OFF_S)[l32][2 * H + p] & live;
                acc = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(f16x4, u32x2{half ? 0u : s, 0u}),
                                                           __builtin_bit_cast(f16x4, u32x2{half ? 0u : q.m & live, 0u}), acc, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = __builtin_fmaf(isum(D0[v]), P0[v], acc[v]);
            asm volatile("" : "+v"(acc), "+v"(q.c1));
            const i32x16 D1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a[1]), __builtin_bit_cast(i32x4, q.c1), magic, 0, 0, 0);
            const f32x16 P1 = scales(dx & second, q.d1 & second & live);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = __builtin_fmaf(isum(D1[v]), P1[v], acc[v]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto add = [&](const f32x16 &acc) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const float t = sum[v] + acc[v];
            if constexpr (NEAR) off[v] += acc[v] - (t - sum[v]);
            sum[v] = t;
        }
    };
    // A chunk that would run past the row's end starts earlier; its blocks in front of `b` count as nothing.
    Chunk k;
    if (b0 < b1) load(k, min(b0, nb - CHUNK));
    for (int b = b0; b < b1; b += CHUNK) {
        const int at = min(b, nb - CHUNK), lo = b - at, hi = min(b1 - at, CHUNK);
        commit(k);
        load(k, min(min(b + CHUNK, b1 - 2), nb - CHUNK));                                // (the last one again)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
        f32x16 acc = zero;
        if (lo < 4) multiply(std::integral_constant<int, 0>{}, lo, hi, acc);
        if (NEAR) { add(acc); acc = zero; }
        if (hi > 4) multiply(std::integral_constant<int, 1>{}, lo, hi, acc);
        add(acc);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // (added as doubles, sum and off apart)
    float *const part = reinterpret_cast<float *>(own);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        part[v * 64 + lane] = sum[v];
        if constexpr (NEAR) part[(16 + v) * 64 + lane] = off[v] == off[v] ? off[v] : 0.f;        // (an infinite sum leaves NaN in off)
    }
    __syncthreads();
    const int64_t row = row_base + l32;
    if (row >= N) return;
    float *__restrict__ y = mat.y;
    if (slice_pairs > 0) y += (size_t)blockIdx.y * (size_t)M * (size_t)mat.ldy;
    // the waves add and store 16 / KS registers' worth each: register v is token 8 * (v / 4) + 4 * half + v % 4
    constexpr int PER = 16 / KS;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int v = wave * PER + i, t = 8 * (v >> 2) + 4 * half + (v & 3);
        double o = 0.;
#pragma unroll
        for (int g = 0; g < KS; g++) {
            const float *p = reinterpret_cast<const float *>(lds + (size_t)g * C::WAVE) + v * 64 + lane;
            o += (double)p[0];
            if constexpr (NEAR) o += (double)p[16 * 64];
        }
        if (t < tokens) y[(size_t)(tok_base + t) * mat.ldy + row] = (float)o * T::POST;
    }
}

template <int WT, int KS, bool NEAR>
hipError_t launch_few(GemmMats mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim, hipStream_t st,
                      int slices, float *part) {
    using C = FewCfg<WT, KS>;
    if ((int64_t)C::LDS > lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_blk32_few_kernel<WT, KS, NEAR>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, C::LDS, lim, grant); e != hipSuccess) return e;
    const TileMap map = make_tile_map(number_row_tiles(mats, 32), ceil_div(M, (int64_t)32), 32 * (8 / KS));
    const GemmMat out = mats.m[0];
    if (slices > 1) { mats.m[0].y = part; mats.m[0].ldy = out.N; }                       // (one matrix)
    hipLaunchKernelGGL(kfn, dim3(map.grid, (unsigned)slices), dim3(64 * KS), C::LDS, st, mats, K, (const uint8_t *)ws, ws_stride, M, map,
                       slices > 1 ? (int)ceil_div(K / 64, (int64_t)slices) : 0);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return slices > 1 ? launch_sum_slices(part, slices, M, out.N, out.y, out.ldy, st, true) : hipSuccess;
}

template <int WT>
hipError_t launch_few_type(int ks, bool near, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim, hipStream_t st,
                           int slices, float *part) {
    switch (ks) {
        case 2: return near ? launch_few<WT, 2, true>(mats, K, ws, ws_stride, M, lim, st, slices, part) : launch_few<WT, 2, false>(mats, K, ws, ws_stride, M, lim, st, slices, part);
        case 4: return near ? launch_few<WT, 4, true>(mats, K, ws, ws_stride, M, lim, st, slices, part) : launch_few<WT, 4, false>(mats, K, ws, ws_stride, M, lim, st, slices, part);
        case 8: return near ? launch_few<WT, 8, true>(mats, K, ws, ws_stride, M, lim, st, slices, part) : launch_few<WT, 8, false>(mats, K, ws, ws_stride, M, lim, st, slices, part);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_gemm_blk32_few(int wtype, int ks, bool near, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim,
                                 hipStream_t st, int slices, float *part) {
    switch (wtype) {
        case T_Q4_0:   return launch_few_type<T_Q4_0>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        case T_Q8_0:   return launch_few_type<T_Q8_0>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        case T_Q5_0:   return launch_few_type<T_Q5_0>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        case T_IQ4_NL: return launch_few_type<T_IQ4_NL>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        case T_Q4_1:   return launch_few_type<T_Q4_1>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        case T_Q5_1:   return launch_few_type<T_Q5_1>(ks, near, mats, K, ws, ws_stride, M, lim, st, slices, part);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace chip
