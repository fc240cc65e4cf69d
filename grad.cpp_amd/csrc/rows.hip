// The many-row projections' variants and the rule that picks one, in a translation unit of
// their own.
#include "rows.h"

#include <stdexcept>
#include <string>

namespace gh {

static void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
}

void split_weights(const float* src, int N, int K, bool gate_up, char* dst, hipStream_t st) {
    const int rows = (N + kSplitPad - 1) / kSplitPad * kSplitPad;
    const size_t chunks = static_cast<size_t>(rows) * (K / 8);
    hipLaunchKernelGGL(split_weights_kernel, dim3(static_cast<unsigned>((chunks + 255) / 256)), dim3(256), 0, st, src, N,
                       K, rows, gate_up ? 1 : 0, dst);
    check(hipGetLastError(), "split_weights");
}

template <bool RMS>
static void norm_split_as(const float* x, const float* gamma, const float* beta, char* out, int M, int d, hipStream_t st) {
    const dim3 grid((M + 15) / 16), block(1024);
    if (d <= 1024) hipLaunchKernelGGL((norm_split_kernel<RMS, 2>), grid, block, 0, st, x, gamma, beta, out, M, d);
    else hipLaunchKernelGGL((norm_split_kernel<RMS, 8>), grid, block, 0, st, x, gamma, beta, out, M, d);
    check(hipGetLastError(), "norm_split");
}

void norm_split(bool rms, const float* x, const float* gamma, const float* beta, char* out, int M, int d, hipStream_t st) {
    if (rms) norm_split_as<true>(x, gamma, beta, out, M, d, st);
    else norm_split_as<false>(x, gamma, beta, out, M, d, st);
}

// Which tiling.  Measured over 16 row counts from 128 to 8192 against six matrices (768 and
// 512 columns: 768, 2304, 4096, 512 outputs; 2048 columns: 768, 512 outputs), the rule takes the
// fastest of the four or one within 7 % of it:
// - While 32 x 32 tiles leave no compute unit with two, they win, and after them 64 x 64 tiles
//   with K over four sets of wavefronts: such a launch is a chain of K steps of about 280 ns
//   each (load, LDS, registers, product), so the shorter chain is what counts (1001 x 768 x
//   2048: 26 us against 39 with K in one set; 100 x 768 x 2048: 13 against 22).
// - With more tiles than compute units the chains hide behind each other.  A compute unit's
//   time per step is 190 ns for a 64 x 64 tile and 624 ns for a 128 x 128 one, which moves half as
//   many operands per product; the cheaper one once tiles are dealt to 256 compute units in
//   whole rounds (4096 x 2304 x 768: 87 us against 95; 8192 x 4096 x 768: 263, i.e. 196 TFLOP/s of
//   fp32 products or 1.18 PFLOP/s of bf16, against 292).
enum Tiling { TILE_32_K4, TILE_64_K4, TILE_64, TILE_128 };

static Tiling pick_tiling(int M, int N) {
    const auto tiles = [&](int t) { return static_cast<long>((M + t - 1) / t) * ((N + t - 1) / t); };
    const auto rounds = [&](int t) { return (tiles(t) + 255) / 256; };
    if (rounds(32) == 1) return TILE_32_K4;
    if (rounds(64) == 1) return TILE_64_K4;
    return rounds(128) > 1 && rounds(128) * 624 < rounds(64) * 190 ? TILE_128 : TILE_64;
}

template <int EPI, int MB, int NB, int WM, int WN, int KG, int STAGES, int PER_CU>
static void launch(SplitGemmParams& p, hipStream_t st) {
    constexpr int TM = 32 * MB * WM, TN = 32 * NB * WN;
    constexpr int lds = (TM + TN) * kSplitRowBytes * STAGES * KG;
    static const hipError_t raised =  // more than the default 64 KB of LDS
        hipFuncSetAttribute(reinterpret_cast<const void*>(split_gemm_kernel<EPI, MB, NB, WM, WN, KG, STAGES, PER_CU>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    check(raised, "hipFuncSetAttribute");
    p.n_tiles = (p.N + TN - 1) / TN;
    p.tiles = (p.M + TM - 1) / TM * p.n_tiles;
    p.nll_stride = p.n_tiles * WN;
    hipLaunchKernelGGL((split_gemm_kernel<EPI, MB, NB, WM, WN, KG, STAGES, PER_CU>), dim3((p.tiles + 7) / 8 * 8),
                       dim3(64 * WM * WN * KG), lds, st, p);
    check(hipGetLastError(), "split_gemm");
}

template <int EPI>
void split_gemm(SplitGemmParams& p, hipStream_t st) {
    switch (pick_tiling(p.M, p.N)) {
        case TILE_32_K4: launch<EPI, 1, 1, 1, 1, 4, 3, 4>(p, st); break;
        case TILE_64_K4: launch<EPI, 1, 1, 2, 2, 4, 3, 1>(p, st); break;
        case TILE_64: launch<EPI, 1, 1, 2, 2, 1, 3, 4>(p, st); break;
        case TILE_128: launch<EPI, 2, 2, 2, 2, 1, 2, 2>(p, st); break;
    }
}

void nll_parts(const SplitGemmParams& p, float* nll, hipStream_t st) {
    hipLaunchKernelGGL(nll_parts_kernel, dim3((p.M + 3) / 4), dim3(256), 0, st, p.nll_part, p.nll_stride, p.nll_target,
                       p.M, p.nll_row0, p.rows_per_seq, p.nll_t0, p.nll_len, nll);
    check(hipGetLastError(), "nll_parts");
}

template void split_gemm<EPI_STORE>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_QKV>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_RESID>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_GELU>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_SWIGLU>(SplitGemmParams&, hipStream_t);

}  // namespace gh
