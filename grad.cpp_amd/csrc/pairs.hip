// The many-row projections in pairs: variants and the rule that picks one, in a translation unit of their own.
#include "rows.h"

#include "kernels_pair.h"

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

constexpr PairOut pair_out(int epilogue) {
    return epilogue == EPI_GELU ? PAIR_GELU : epilogue == EPI_SWIGLU ? PAIR_SWIGLU : epilogue == EPI_STORE ? PAIR_LOGITS : PAIR_ROWS;
}

template <int EPI>
void pair_gemm(SplitGemmParams& p, hipStream_t st) {
    const PairTiling tiling = pair_tiling(p.M, p.N, p.K, pair_out(EPI));
    if constexpr (EPI != EPI_STORE) {
        if (tiling == PAIR_MIXED) return launch_mixed<EPI>(p, st);
    }
    switch (tiling) {
        case PAIR_128: launch<EPI, 2, 2, 2, 2, 1, 2>(p, st); break;
        case PAIR_128x64: launch<EPI, 2, 1, 2, 2, 1, 2>(p, st); break;
        case PAIR_64: launch<EPI, 1, 1, 2, 2, 1, 4>(p, st); break;
        case PAIR_64_K2: launch<EPI, 1, 1, 2, 2, 2, 2>(p, st); break;
        case PAIR_64x96_K2: launch<EPI, 1, 3, 2, 1, 2, 2>(p, st); break;
        case PAIR_64x96_K4: launch<EPI, 1, 3, 2, 1, 4, 1>(p, st); break;
        case PAIR_32_K4: launch<EPI, 1, 1, 1, 1, 4, 2>(p, st); break;
        case PAIR_MIXED: throw std::logic_error("pair_gemm: tiles in quarters have no scored logits");
    }
}

template void pair_gemm<EPI_STORE>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_QKV>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_RESID>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_GELU>(SplitGemmParams&, hipStream_t);
template void pair_gemm<EPI_SWIGLU>(SplitGemmParams&, hipStream_t);

}  // namespace gh
