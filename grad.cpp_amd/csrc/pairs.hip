// The many-row projections in pairs: variants and the rule that picks one, in a translation unit of their own.
#include "rows.h"

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

enum Tiling { TILE_32_K4, TILE_64_K4, TILE_64, TILE_128x64, TILE_128 };

static Tiling pick_tiling(int M, int N, int K) {
    const auto tiles = [&](int t) { return static_cast<long>((M + t - 1) / t) * ((N + t - 1) / t); };
    const auto rounds = [&](int t) { return (tiles(t) + 255) / 256; };
    if (K % 256 == 0) {
        if (rounds(32) <= 2) return TILE_32_K4;
        if (rounds(64) == 1) return TILE_64_K4;
    }
    const long tall = static_cast<long>((M + 127) / 128) * ((N + 63) / 64);
    if (rounds(64) == 2 && tall <= 256 && K >= 768) return TILE_128x64;
    return rounds(128) * 28 < rounds(64) * 10 ? TILE_128 : TILE_64;
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
void pair_gemm(SplitGemmParams& p, hipStream_t st) {
    switch (pick_tiling(p.M, p.N, p.K)) {
        case TILE_32_K4: launch<EPI, 1, 1, 1, 1, 4, 2>(p, st); break;
        case TILE_64_K4: launch<EPI, 1, 1, 2, 2, 4, 1>(p, st); break;
        case TILE_64: launch<EPI, 1, 1, 2, 2, 1, 4>(p, st); break;
        case TILE_128x64: launch<EPI, 2, 1, 2, 2, 1, 2>(p, st); break;
        case TILE_128: launch<EPI, 2, 2, 2, 2, 1, 2>(p, st); break;
    }
}

template void pair_gemm<EPI_STORE>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_QKV>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_RESID>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_GELU>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_SWIGLU>(SplitGemmParams&, hipStream_t);

}  // namespace gh
