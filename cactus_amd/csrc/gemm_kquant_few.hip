// GEMM for gfx950 over K-quant weights (Q2_K .. Q6_K, IQ4_XS) and Q8_K activations for products of few tokens: the batched form of
// lm_ggml_vec_dot_q2_K_q8_K .. _q6_K_q8_K, _iq4_xs_q8_K (reference ggml-cpu/ggml-cpu-quants.c) as driven by
// lm_ggml_compute_forward_mul_mat (ggml-cpu/ggml-cpu.c:1257-1449).
//
// The waves of a workgroup share one tile of 16 rows x 16 TT tokens and deal its super-blocks out between them.  Each is on its own until the
// end: it loads its rows' packed bytes and its tokens' quants in memory order, a super-block ahead of the one it multiplies, turns them round
// through a stretch of LDS of its own, with no barrier, and expands its lanes' operands in registers (kquant_rows_dev.h; what the digit planes
// are: gemm_kquant_rows.hip).  A v_mfma_i32_16x16x64_i8 covers two k-blocks: lane (x, g) holds the k-half g % 2 of a k-block of item (H, g / 2), for rows
// and tokens alike.  The waves' sums meet in LDS once and are added as doubles.  A wave scales and adds its super-blocks in 32 bits, at most eight of
// them (kq_few_plan), no further from the 64-bit sums than the GEMV, the walks and the slices of K that ran before (2-norm of the error over 239 random
// products of Q4_K, Q5_K, Q6_K and Q3_K, 1024 to 14336 values at 5 to 300 tokens: 0.80 of theirs on average, 1.05 at most, where the sample is good for
// 0.03); but rows of up to three super-blocks, and Q2_K and IQ4_XS, whose slices were short chains added as doubles, in 64 bits, a result rounded once:
// in 32 bits they were up to 1.16 and 1.07 x as far (512 values at 15 tokens, GEMV / 32 bits / 64: Q3_K 4.0e-8 / 4.5e-8 / 2.7e-8).  64 bits
// take 1.025 x the time (83 products of Q2_K and IQ4_XS; so does the product in 32 bits added in 64).
//
// Bound: the issue of vector instructions (by the counters 214 per super-block of 16 rows x 16 tokens for Q4_K, 267 to 291 for Q6_K, over half of them the expansion) at two
// to four waves a SIMD, and the tokens' quants, 4 KB for the 1.3 to 3.4 KB of 16 rows: tiles of 32 rows halve those where there are rows enough.  us, what ran
// before / this, 8 tokens (a GEMV): Q6_K 4096 values x 4096 rows 9.6 / 7.7, 14336 x 4096 20.0 / 16.5, 4096 x 32000 37 / 31; Q4_K 1024 x 3072 7.7 / 4.1; 32
// tokens (the GEMM, in slices of K): Q4_K 4096 x 4096 13.8 / 8.3, x 14336 27.0 / 18.7, 2048 x 768 11.2 / 5.1; 64 tokens Q4_K 4096 x 4096
// 16.1 / 11.1.  16 rows rather than 32 a tile because 4096 rows are then a workgroup for every CU; more waves than super-blocks have nothing to share.
#include "dev_common.h"
#include "act_layout.h"
#include "kernels.h"
#include "kquant_rows_dev.h"
#include <algorithm>
#include <type_traits>

namespace chip {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// Rows of up to three super-blocks, and Q2_K and IQ4_XS of any length, are scaled and added in 64 bits.
constexpr int FEW_SHORT = 3;
constexpr bool few_always_wide(int wt) { return wt == T_Q2_K || wt == T_IQ4_XS; }

template <int WT, int RT, int TT>
struct KfCfg {
    using T = KR<WT>;
    static constexpr int BM = 16 * RT, BN = 16 * TT;
    static constexpr int NLD = (BM * T::NCH + 63) / 64, NX = BN / 4;      // loads of a lane: weights, tokens' quants
    static constexpr int ROW = T::NCH | 1;                                // cells a row takes in LDS: 16 rows' cells of one index in different banks
    // a wave's stretch: rows, tokens' quants ([token][16 cells], swizzled), their scales, their block sums as fp16 ([token][16])
    static constexpr int OFF_X = BM * ROW * 16, OFF_D = OFF_X + BN * 256, OFF_S = OFF_D + BN * 4, WAVE = OFF_S + (T::NF16 ? BN * 32 : 0);
    static_assert(WAVE % 16 == 0 && WAVE >= BM * BN * 8, "a wave's sums take the place of its operands");
};

// One tile; `stretch`: bytes of LDS a wave has.  WIDE: super-blocks are scaled and added in 64 bits.
template <int WT, int RT, int TT, bool WIDE>
__device__ __forceinline__ void few_tile(uint8_t *lds, int stretch, const GemmMat &mat, int row_tile, int tok_tile, int64_t K,
                                         const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M) {
    using T = KR<WT>;
    using C = KfCfg<WT, RT, TT>;
    using real = std::conditional_t<WIDE, double, float>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ks = (int)blockDim.x >> 6;
    const int x = lane & 15, g = lane >> 4, hf = g & 1, p = g >> 1;
    const int64_t N = mat.N, row_base = (int64_t)row_tile * C::BM, tok_base = (int64_t)tok_tile * C::BN;
    const int tokens = (int)min((int64_t)C::BN, M - tok_base), nsb = (int)(K / QK_K);
    uint8_t *const own = lds + wave * stretch;

    // (offsets of 32 bits from the tile's first row and first token: kq_few_plan, and few_group for members that share a launch, see to it)
    const uint8_t *const w0 = mat.W + (size_t)row_base * mat.nb01, *const x0 = ws + (size_t)tok_base * ws_stride;
    uint32_t woff[C::NLD], wdst[C::NLD], xoff[C::NX];
#pragma unroll
    for (int t = 0; t < C::NLD; t++) {
        const int i = min(lane + 64 * t, C::BM * T::NCH - 1), r = i / T::NCH, c = i % T::NCH;
        woff[t] = (uint32_t)min((int64_t)r, N - 1 - row_base) * (uint32_t)mat.nb01 + (uint32_t)(c == T::NCH - 1 ? T::BYTES - 16 : 16 * c);
        wdst[t] = (uint32_t)(r * C::ROW + c);
    }
#pragma unroll
    for (int t = 0; t < C::NX; t++) xoff[t] = (uint32_t)min(4 * t + g, tokens - 1) * (uint32_t)ws_stride + 16u * x;
    const uint32_t doff = (uint32_t)min(lane & (C::BN - 1), tokens - 1) * (uint32_t)ws_stride + (uint32_t)q8_K_off_d(K);
    const uint32_t soff = (uint32_t)min((lane >> 1) & (C::BN - 1), tokens - 1) * (uint32_t)ws_stride + (uint32_t)q8_K_off_bsums(K) + 16u * (lane & 1);

    struct Load {
        u32x4 w[C::NLD], x[C::NX], s;
        float d;
    };
    auto load = [&](Load &k, int sb) {
#pragma unroll
        for (int t = 0; t < C::NLD; t++) k.w[t] = *reinterpret_cast<const typename T::chunk_t *>(w0 + (size_t)sb * T::BYTES + woff[t]);
#pragma unroll
        for (int t = 0; t < C::NX; t++) k.x[t] = *reinterpret_cast<const u32x4 *>(x0 + (size_t)sb * QK_K + xoff[t]);
        k.d = *reinterpret_cast<const float *>(x0 + 4 * (size_t)sb + doff);
        if constexpr (T::NF16 > 0) k.s = *reinterpret_cast<const u32x4_a4 *>(x0 + 32 * (size_t)sb + soff);
    };
    auto commit = [&](const Load &k) {
#pragma unroll
        for (int t = 0; t < C::NLD; t++) reinterpret_cast<u32x4 *>(own)[wdst[t]] = k.w[t];
#pragma unroll
        for (int t = 0; t < C::NX; t++) {
            const int tok = 4 * t + g;
            reinterpret_cast<u32x4 *>(own + C::OFF_X)[tok * 16 + (x ^ (tok & 15))] = k.x[t];
        }
        if (lane < C::BN) reinterpret_cast<float *>(own + C::OFF_D)[lane] = k.d;
        if constexpr (T::NF16 > 0)
            if (lane < 2 * C::BN) reinterpret_cast<u32x4 *>(own + C::OFF_S)[lane] = i16x8_to_f16(k.s);
    };

    const u32x4 *const row = reinterpret_cast<const u32x4 *>(own) + x * C::ROW;           // and 16 rows on per tile of rows
    // cell 2 * k-block + k-half of the lane's token; the bits that H and the second k-block add are not set in it
    const uint32_t b_lane = (uint32_t)C::OFF_X + (uint32_t)x * 256u + 16u * (uint32_t)((2 * (3 - T::NEXT) * p + hf) ^ x);
    real out[RT][TT][4] = {};

    Load k;
    load(k, wave);                                                                       // (ks <= nsb: launch_few)
    for (int sb = wave; sb < nsb; sb += ks) {
        commit(k);
        if (sb + ks < nsb) load(k, sb + ks);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // (beside 64-bit sums the headers of all row tiles and a half's quants would not fit the registers: they are read where they are used)
        typename T::Hdr held[RT];
        auto hdr = [&](int r) { return WIDE ? T::hdr(row + 16 * r * C::ROW, hf) : held[r]; };
        auto quants = [&](int H, int e, int c) { return *reinterpret_cast<const u32x4 *>(own + c * 4096 + (b_lane ^ (uint32_t)(16 * (8 * H + 2 * T::NEXT * e)))); };
        if constexpr (!WIDE)
#pragma unroll
            for (int r = 0; r < RT; r++) held[r] = T::hdr(row + 16 * r * C::ROW, hf);
        i32x4 P[T::NPL][RT][TT];
#pragma unroll
        for (int H = 0; H < 2; H++) {
            if constexpr (WT == T_Q5_K && WIDE) asm volatile("" ::: "memory");            // its header again for each half and for the fold
            u32x4 a[2][TT];
            if constexpr (!WIDE)
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int c = 0; c < TT; c++) a[e][c] = quants(H, e, c);
#pragma unroll
            for (int r = 0; r < RT; r++) {
                u32x4 w[2][T::NPL];
                T::expand(T::load(row + 16 * r * C::ROW, H, p, hf), hdr(r), H, p, hf, w);
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int c = 0; c < TT; c++) {
                        if constexpr (WIDE) a[e][c] = quants(H, e, c);
#pragma unroll
                        for (int pl = 0; pl < T::NPL; pl++)
                            P[pl][r][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a[e][c]), __builtin_bit_cast(i32x4, w[e][pl]),
                                                                                H == 0 && e == 0 ? i32x4{0, 0, 0, 0} : P[pl][r][c], 0, 0, 0);
                    }
            }
        }
        // fold, as the reference does once per super-block: out += dx * (d * sumi - dmin * summ)
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if constexpr (WT == T_Q5_K && WIDE) asm volatile("" ::: "memory");
            const uint32_t scales = T::scales(hdr(r));
            real d = h2f(scales), dmin = h2f(scales >> 16);
            if constexpr (!WIDE) asm volatile("" : "+v"(d), "+v"(dmin));   // widened once: as halves they would make the multiply-adds half-rate mixed ones
#pragma unroll
            for (int c = 0; c < TT; c++) {
                f32x4 F = {0.f, 0.f, 0.f, 0.f};
                if constexpr (T::NF16 > 0) {
                    const u32x2 s = *reinterpret_cast<const u32x2 *>(own + C::OFF_S + (16 * c + x) * 32 + 8 * g);
                    F = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, s), __builtin_bit_cast(f16x4, T::f16_quad(row + 16 * r * C::ROW, g)), F, 0, 0, 0);
                }
                const f32x4 dx = *reinterpret_cast<const f32x4 *>(own + C::OFF_D + (16 * c + 4 * g) * 4);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float f[2] = {F[v], 0.f};
                    out[r][c][v] = mul_add(T::value(P[0][r][c][v], P[T::NPL - 1][r][c][v], f, d, dmin), (real)dx[v], out[r][c][v]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // register v of tile (r, c) is token 16 c + 4 g + v, the lane's x its row 16 r + x
    real *const part = reinterpret_cast<real *>(own);
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int c = 0; c < TT; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) part[((c * RT + r) * 4 + v) * 64 + lane] = out[r][c][v];
    __syncthreads();
    for (int e = threadIdx.x; e < 256 * RT * TT; e += (int)blockDim.x) {
        double o = 0.;
        for (int w = 0; w < ks; w++) o += (double)reinterpret_cast<const real *>(lds + w * stretch)[e];
        const int tile = e >> 8, t = 16 * (tile / RT) + 4 * ((e & 63) >> 4) + ((e >> 6) & 3);
        const int64_t r = row_base + 16 * (tile % RT) + (e & 15);
        if (t < tokens && r < N) mat.y[(size_t)(tok_base + t) * mat.ldy + r] = (float)o;
    }
}

constexpr int few_waves(int rt, int tt) { return rt * tt == 1 ? 16 : 8; }               // most waves of a workgroup
#define KQ_FEW_BOUNDS(RT, TT) __launch_bounds__(64 * few_waves(RT, TT)) __attribute__((amdgpu_waves_per_eu((RT) * (TT) == 1 ? 4 : (RT) * (TT) == 2 ? 3 : 2)))

template <int WT, int RT, int TT, bool WIDE>
__global__ KQ_FEW_BOUNDS(RT, TT)
void gemm_kq_few_kernel(GemmMats mats, int64_t K, const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M, TileMap map) {
    extern __shared__ __align__(16) uint8_t lds[];
    TileCoord tc = xcd_tile(blockIdx.x, map);
    if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;            // padding of the tile map
    const GemmMat mat = pick_gemm_mat(mats, tc.row_tile);
    few_tile<WT, RT, TT, WIDE>(lds, KfCfg<WT, RT, TT>::WAVE, mat, tc.row_tile, tc.tok_tile, K, ws, ws_stride, M);
}

// matrices of two types on the same rows: the row tiles from `second` on are of type WB
template <int WA, int WB, int TT> constexpr int few_two_stretch() { return KfCfg<WA, 1, TT>::WAVE > KfCfg<WB, 1, TT>::WAVE ? KfCfg<WA, 1, TT>::WAVE : KfCfg<WB, 1, TT>::WAVE; }
template <int WA, int WB, int TT, bool SHORT>
__global__ KQ_FEW_BOUNDS(1, TT)
void gemm_kq_few_two_kernel(GemmMats mats, int second, int64_t K, const uint8_t *__restrict__ ws, size_t ws_stride, int64_t M, TileMap map) {
    extern __shared__ __align__(16) uint8_t lds[];
    TileCoord tc = xcd_tile(blockIdx.x, map);
    if (tc.row_tile >= map.row_tiles || tc.tok_tile >= map.tok_tiles) return;
    constexpr int STRETCH = few_two_stretch<WA, WB, TT>();
    const bool of_b = tc.row_tile >= second;
    const GemmMat mat = pick_gemm_mat(mats, tc.row_tile);
    if (of_b) few_tile<WB, 1, TT, SHORT || few_always_wide(WB)>(lds, STRETCH, mat, tc.row_tile, tc.tok_tile, K, ws, ws_stride, M);
    else few_tile<WA, 1, TT, SHORT || few_always_wide(WA)>(lds, STRETCH, mat, tc.row_tile, tc.tok_tile, K, ws, ws_stride, M);
}

struct FewCall { GemmMats mats; int64_t K; const void *ws; size_t ws_stride; int64_t M; const DeviceLimits &lim; hipStream_t st; int ks; };

template <int WT, int RT, int TT, bool WIDE>
hipError_t launch_few(FewCall c) {
    using C = KfCfg<WT, RT, TT>;
    const size_t bytes = (size_t)c.ks * C::WAVE;
    if (c.ks < 1 || c.ks > few_waves(RT, TT) || c.ks > c.K / QK_K || (int64_t)bytes > c.lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kq_few_kernel<WT, RT, TT, WIDE>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, bytes, c.lim, grant); e != hipSuccess) return e;
    const TileMap map = make_tile_map(number_row_tiles(c.mats, C::BM), ceil_div(c.M, (int64_t)C::BN), 32 * std::max(1, 16 / c.ks));
    hipLaunchKernelGGL(kfn, dim3(map.grid), dim3(64 * c.ks), bytes, c.st, c.mats, c.K, (const uint8_t *)c.ws, c.ws_stride, c.M, map);
    return hipGetLastError();
}
template <int WA, int WB, int TT, bool SHORT>
hipError_t launch_two(FewCall c, int first_b) {
    const size_t bytes = (size_t)c.ks * few_two_stretch<WA, WB, TT>();
    if (c.ks < 1 || c.ks > few_waves(1, TT) || c.ks > c.K / QK_K || (int64_t)bytes > c.lim.max_lds_per_block) return hipErrorInvalidValue;
    auto kfn = gemm_kq_few_two_kernel<WA, WB, TT, SHORT>;
    static LdsGrant grant;
    if (hipError_t e = grant_dynamic_lds(kfn, bytes, c.lim, grant); e != hipSuccess) return e;
    const TileMap map = make_tile_map(number_row_tiles(c.mats, 16), ceil_div(c.M, (int64_t)(16 * TT)), 32 * std::max(1, 16 / c.ks));
    hipLaunchKernelGGL(kfn, dim3(map.grid), dim3(64 * c.ks), bytes, c.st, c.mats, c.mats.first[first_b], c.K, (const uint8_t *)c.ws, c.ws_stride, c.M, map);
    return hipGetLastError();
}

template <int WT, bool WIDE>
hipError_t launch_few_form(int rt, int tt, const FewCall &c) {
    if (rt == 1) return tt == 1 ? launch_few<WT, 1, 1, WIDE>(c) : launch_few<WT, 1, 2, WIDE>(c);
    return tt == 1 ? launch_few<WT, 2, 1, WIDE>(c) : launch_few<WT, 2, 2, WIDE>(c);
}
bool few_short(const FewCall &c) { return c.K <= FEW_SHORT * QK_K; }
template <int WT>
hipError_t launch_few_type(int rt, int tt, const FewCall &c) {
    if (few_always_wide(WT) || few_short(c)) return launch_few_form<WT, true>(rt, tt, c);
    return launch_few_form<WT, few_always_wide(WT)>(rt, tt, c);
}
template <int WA, int WB, int TT>
hipError_t launch_two_form(const FewCall &c, int first_b) {
    return few_short(c) ? launch_two<WA, WB, TT, true>(c, first_b) : launch_two<WA, WB, TT, false>(c, first_b);
}
template <int WA, int WB>
hipError_t launch_two_types(int tt, const FewCall &c, int first_b) {
    if constexpr (WA < WB) return tt == 1 ? launch_two_form<WA, WB, 1>(c, first_b) : launch_two_form<WA, WB, 2>(c, first_b);
    return hipErrorInvalidValue;
}
template <int WA>
hipError_t launch_two_types(int wb, int tt, const FewCall &c, int first_b) {
    switch (wb) {
        case T_Q3_K: return launch_two_types<WA, T_Q3_K>(tt, c, first_b);
        case T_Q4_K: return launch_two_types<WA, T_Q4_K>(tt, c, first_b);
        case T_Q5_K: return launch_two_types<WA, T_Q5_K>(tt, c, first_b);
        case T_Q6_K: return launch_two_types<WA, T_Q6_K>(tt, c, first_b);
        case T_IQ4_XS: return launch_two_types<WA, T_IQ4_XS>(tt, c, first_b);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int gemm_kq_few_stretch(int wtype, int rt, int tt) {
    auto of = [&](auto t) {
        constexpr int WT = decltype(t)::value;
        return rt == 1 ? (tt == 1 ? KfCfg<WT, 1, 1>::WAVE : KfCfg<WT, 1, 2>::WAVE) : (tt == 1 ? KfCfg<WT, 2, 1>::WAVE : KfCfg<WT, 2, 2>::WAVE);
    };
    switch (wtype) {
        case T_Q4_K: return of(std::integral_constant<int, T_Q4_K>{});
        case T_Q5_K: return of(std::integral_constant<int, T_Q5_K>{});
        case T_Q6_K: return of(std::integral_constant<int, T_Q6_K>{});
        case T_Q3_K: return of(std::integral_constant<int, T_Q3_K>{});
        case T_Q2_K: return of(std::integral_constant<int, T_Q2_K>{});
        default:     return of(std::integral_constant<int, T_IQ4_XS>{});
    }
}

// types[i]: the type of mats.m[i]; of two types the lower id stands first (f.rt is 1 then).
hipError_t launch_gemm_kq_few(KqFew f, const int *types, const GemmMats &mats, int64_t K, const void *ws, size_t ws_stride, int64_t M, const DeviceLimits &lim,
                              hipStream_t st) {
    const FewCall c{mats, K, ws, ws_stride, M, lim, st, f.ks};
    int first_b = 1;
    while (first_b < mats.count && types[first_b] == types[0]) first_b++;
    if (first_b < mats.count) {
        switch (types[0]) {
            case T_Q2_K: return launch_two_types<T_Q2_K>(types[first_b], f.tt, c, first_b);
            case T_Q3_K: return launch_two_types<T_Q3_K>(types[first_b], f.tt, c, first_b);
            case T_Q4_K: return launch_two_types<T_Q4_K>(types[first_b], f.tt, c, first_b);
            case T_Q5_K: return launch_two_types<T_Q5_K>(types[first_b], f.tt, c, first_b);
            case T_Q6_K: return launch_two_types<T_Q6_K>(types[first_b], f.tt, c, first_b);
            default: return hipErrorInvalidValue;
        }
    }
    switch (types[0]) {
        case T_Q4_K: return launch_few_type<T_Q4_K>(f.rt, f.tt, c);
        case T_Q5_K: return launch_few_type<T_Q5_K>(f.rt, f.tt, c);
        case T_Q6_K: return launch_few_type<T_Q6_K>(f.rt, f.tt, c);
        case T_Q3_K: return launch_few_type<T_Q3_K>(f.rt, f.tt, c);
        case T_Q2_K: return launch_few_type<T_Q2_K>(f.rt, f.tt, c);
        case T_IQ4_XS: return launch_few_type<T_IQ4_XS>(f.rt, f.tt, c);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace chip
