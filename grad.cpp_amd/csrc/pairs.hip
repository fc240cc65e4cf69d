// The many-row projections in pairs: variants and the rule that picks one, in a translation unit of their own.
#include "rows.h"

#include "kernels_pair.h"

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <string>

namespace gh {

static void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
}

void pair_weights(const float* src, int N, int K, bool gate_up, char* dst, float* unit, float* norm, hipStream_t st) {
    const int rows = static_cast<int>(pair_rows(N));
    hipLaunchKernelGGL(pair_weights_kernel, dim3(rows / 4), dim3(256), 0, st, src, N, K, rows, gate_up ? 1 : 0, dst, unit, norm);
    check(hipGetLastError(), "pair_weights");
}

template <bool RMS>
static void norm_pair_as(const float* x, const float* gamma, const float* beta, char* out, int M, int d, float pair_scale,
                         hipStream_t st) {
    const dim3 grid((M + 15) / 16), block(1024);
    if (d <= 1024) hipLaunchKernelGGL((norm_pair_kernel<RMS, 2>), grid, block, 0, st, x, gamma, beta, out, M, d, pair_scale);
    else if (d <= 4096) hipLaunchKernelGGL((norm_pair_kernel<RMS, 8>), grid, block, 0, st, x, gamma, beta, out, M, d, pair_scale);
    else hipLaunchKernelGGL((norm_pair_long_kernel<RMS>), grid, block, 0, st, x, gamma, beta, out, M, d, pair_scale);
    check(hipGetLastError(), "norm_pair");
}

void norm_pair(bool rms, const float* x, const float* gamma, const float* beta, char* out, int M, int d, float pair_scale,
               hipStream_t st) {
    if (rms) norm_pair_as<true>(x, gamma, beta, out, M, d, pair_scale, st);
    else norm_pair_as<false>(x, gamma, beta, out, M, d, pair_scale, st);
}

// The tilings, and what a launch takes with each: with n tiles on the fullest of 256 compute units and K in thousands
//   start + max(chain K, n step K) + n out
// us, fitted to 230 launches (160 to 16384 rows against the ten matrices of models 512 and 768 columns wide: W_o, QKV,
// both FFN1 and FFN2), medians off by 2 to 5 %.  A lone workgroup is a chain of K steps (64 x 64 tiles with K shared by
// two sets of wavefronts, and 32 x 32 ones by four, are the shorter chains); beside others its chain hides, and what
// counts is what the unit moves through LDS and multiplies; `out` is the epilogue, of a residual (queries, keys, values
// and logits counted like it), a GELU or a SwiGLU.  Taking the least by this rule, those launches take 0.8 % longer
// than with the best of the seven tilings each (at most 18 %), by the three-part form's rule 5.1 (at most 44 %): 1999 x
// 768 x 768 14.0 -> 11.4 us, 1999 x 768 x 2048 31.9 -> 24.2, 1999 x 2304 x 768 31.8 -> 31.1, 1999 x 3072 x 768 37.5 ->
// 34.8.  (Four tilings more, among them 96 x 192, 192 x 64 and 128 x 96, were the best by less than 1 % together.)
struct Tiling {
    int m, n, sets;  // rows, outputs, sets of wavefronts that share K
    float start, chain, step, out[3];
};
enum { TILE_128, TILE_128x64, TILE_64, TILE_64_K2, TILE_64x96_K2, TILE_64x96_K4, TILE_32_K4, TILINGS, TILE_MIXED = TILINGS };
constexpr Tiling kTilings[TILINGS] = {
    {128, 128, 1, 1.64f, 21.42f, 18.17f, {4.43f, 4.01f, 3.31f}}, {128, 64, 1, 2.15f, 13.10f, 10.78f, {1.94f, 1.80f, 1.20f}},
    {64, 64, 1, 1.90f, 9.58f, 6.45f, {1.00f, 0.80f, 0.58f}},     {64, 64, 2, 1.61f, 6.59f, 6.31f, {1.18f, 1.18f, 1.01f}},
    {64, 96, 2, 2.37f, 10.21f, 8.57f, {2.15f, 2.14f, 1.44f}},    {64, 96, 4, 0.50f, 2.40f, 8.44f, {3.72f, 4.87f, 3.85f}},
    {32, 32, 4, 2.14f, 2.68f, 2.53f, {0.46f, 0.81f, 0.62f}},
};

// TILE_MIXED: 128 x 128 tiles in whole rounds of 256 and the rest, at most 64 of them, as 64 x 64 quarters in the same
// launch, at most one for each compute unit, beside its last whole tile (both fit it).  2000 x 2304 outputs are 288
// tiles: 32 compute units had two and the others waited.  Of 230 launches (160 to 16384 rows) the rule gives it 18, all
// of them faster than what they took before, by 7 to 22 % (1999 x 2304 x 768 33.0 -> 28.6 us, in a prompt 37.5 -> 32.4,
// 6000 x 768 x 2048 67.8 -> 61.3, 1280 x 4096 x 768 32.2 -> 27.1, 7000 x 3072 x 768 111.0 -> 101.3); with more than one
// quarter for a compute unit it is the slower one in 32 of 45 (2600 x 3072 x 768 42.4 -> 48.6, 1800 x 4096 x 768 38.2
// -> 44.0).  Not for scored logits, whose sums of exponentials are kept for 64 columns at a time.
constexpr int kMixedRest = 64;

static int pick_tiling(int M, int N, int K, int epilogue) {
    const int out = epilogue == EPI_GELU ? 1 : epilogue == EPI_SWIGLU ? 2 : 0;
    int best = TILE_128;
    float least = INFINITY;
    for (int i = 0; i < TILINGS; i++) {
        const Tiling& t = kTilings[i];
        if (K % (64 * t.sets) != 0) continue;  // (whole parts per set)
        const float tiles = static_cast<float>((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n), n = std::ceil(tiles / 256.0f);
        const float us = t.start + std::max(t.chain, n * t.step) * K * 1e-3f + n * t.out[out];
        if (us < least) {
            least = us;
            best = i;
        }
    }
    const int tiles = (M + 127) / 128 * ((N + 127) / 128), rounds = tiles / 256, rest = tiles % 256;
    if (epilogue != EPI_STORE && rounds > 0 && rest > 0 && rest <= kMixedRest) {
        const Tiling &a = kTilings[TILE_128], &b = kTilings[TILE_64];
        const float us = a.start + std::max(a.chain, rounds * a.step + b.step) * K * 1e-3f + rounds * a.out[out] + b.out[out];
        if (us < least) best = TILE_MIXED;
    }
    return best;
}

template <int EPI, int MB, int NB, int WM, int WN, int KG, int PER_CU>
static void launch(SplitGemmParams& p, hipStream_t st) {
    constexpr int TM = 32 * MB * WM, TN = 32 * NB * WN;
    constexpr int lds = (TM + TN) / 16 * 1024 * kPairStages * KG;
    static const hipError_t raised =  // more than the default 64 KB of LDS
        hipFuncSetAttribute(reinterpret_cast<const void*>(pair_gemm_kernel<EPI, MB, NB, WM, WN, KG, PER_CU>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    check(raised, "hipFuncSetAttribute");
    p.n_tiles = (p.N + TN - 1) / TN;
    p.tiles = (p.M + TM - 1) / TM * p.n_tiles;
    p.nll_stride = p.n_tiles * WN;
    hipLaunchKernelGGL((pair_gemm_kernel<EPI, MB, NB, WM, WN, KG, PER_CU>), dim3((p.tiles + 7) / 8 * 8), dim3(64 * WM * WN * KG),
                       lds, st, p);
    check(hipGetLastError(), "pair_gemm");
}

template <int EPI>
static void launch_mixed(SplitGemmParams& p, hipStream_t st) {
    constexpr int lds = (128 + 128) / 16 * 1024 * kPairStages;
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(pair_mixed_kernel<EPI>),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    check(raised, "hipFuncSetAttribute");
    p.n_tiles = (p.N + 127) / 128;
    p.tiles = (p.M + 127) / 128 * p.n_tiles;
    const int whole = p.tiles / 256 * 256, rest = p.tiles - whole;
    hipLaunchKernelGGL((pair_mixed_kernel<EPI>), dim3(whole + (rest + 7) / 8 * 8 * 4), dim3(256), lds, st, p, whole);
    check(hipGetLastError(), "pair_gemm");
}

template <int EPI>
void pair_gemm(SplitGemmParams& p, hipStream_t st) {
    const int tiling = pick_tiling(p.M, p.N, p.K, EPI);
    if constexpr (EPI != EPI_STORE) {
        if (tiling == TILE_MIXED) return launch_mixed<EPI>(p, st);
    }
    switch (tiling) {
        case TILE_128: launch<EPI, 2, 2, 2, 2, 1, 2>(p, st); break;
        case TILE_128x64: launch<EPI, 2, 1, 2, 2, 1, 2>(p, st); break;
        case TILE_64: launch<EPI, 1, 1, 2, 2, 1, 4>(p, st); break;
        case TILE_64_K2: launch<EPI, 1, 1, 2, 2, 2, 2>(p, st); break;
        case TILE_64x96_K2: launch<EPI, 1, 3, 2, 1, 2, 2>(p, st); break;
        case TILE_64x96_K4: launch<EPI, 1, 3, 2, 1, 4, 1>(p, st); break;
        case TILE_32_K4: launch<EPI, 1, 1, 1, 1, 4, 2>(p, st); break;
    }
}

template void pair_gemm<EPI_STORE>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_QKV>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_RESID>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_GELU>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_SWIGLU>(SplitGemmParams&, hipStream_t);

}  // namespace gh
