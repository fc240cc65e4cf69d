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

// A workgroup per run.  The value of a rank is found byte by byte of the magnitudes' bits, which are in the order of the
// magnitudes: of those that agree with what is known so far, how many have each next byte.  Bound by five dependent passes over
// a run, out of the L2 but for the first: 12 to 37 us for a layer's runs of 512 to 4096 values.  With the vectors copied to the host
// one by one and the ranks found there, the first pass of 700 rows of a model took 3.6 ms (Llama block, 8 layers of 768
// columns), 2.5 (GPT-2, 6 of 512) and 10.0 (32 of 512); now 1.8, 1.0 and 4.3.
constexpr int kSizesThreads = 1024;

static __global__ __launch_bounds__(kSizesThreads) void sizes_kernel(const SizeRuns runs, Sizes* out) {
    __shared__ unsigned count[256], nan_or_top[2], rank_and_bits[2];
    const int n = runs.n[blockIdx.x];
    const unsigned* const v = reinterpret_cast<const unsigned*>(runs.at[blockIdx.x]);
    constexpr unsigned kInf = 0x7f800000u;
    if (threadIdx.x < 2) nan_or_top[threadIdx.x] = rank_and_bits[threadIdx.x] = 0;
    __syncthreads();
    unsigned top = 0, nan = 0, some = 0;
    for (int i = threadIdx.x; i < n; i += kSizesThreads) {
        const unsigned bits = v[i] & 0x7fffffffu;
        if (bits > kInf) nan = 1;
        else top = max(top, bits), some += bits != 0;
    }
    if (nan) atomicOr(&nan_or_top[0], 1u);
    atomicMax(&nan_or_top[1], top);
    atomicAdd(&rank_and_bits[0], some);
    __syncthreads();
    if (threadIdx.x == 0) rank_and_bits[0] /= 8;  // from the smallest of those that are not zero
    for (int shift = 24; shift >= 0; shift -= 8) {
        if (threadIdx.x < 256) count[threadIdx.x] = 0;
        __syncthreads();
        const unsigned known = rank_and_bits[1];
        for (int i = threadIdx.x; i < n; i += kSizesThreads) {
            const unsigned bits = v[i] & 0x7fffffffu;
            if (bits != 0 && bits <= kInf && (shift == 24 || (bits ^ known) >> (shift + 8) == 0)) atomicAdd(&count[bits >> shift & 255], 1u);
        }
        __syncthreads();
        if (threadIdx.x < 64) {  // (four bytes to a lane; with no value at all none of them holds the rank)
            const unsigned rank = rank_and_bits[0];
            unsigned mine = 0, upto;
            for (int i = 0; i < 4; i++) mine += count[4 * threadIdx.x + i];
            upto = mine;
            for (int far = 1; far < 64; far *= 2) {
                const unsigned below = __shfl_up(upto, far, 64);
                if (threadIdx.x >= static_cast<unsigned>(far)) upto += below;
            }
            unsigned left = rank - (upto - mine), byte = 4 * threadIdx.x;
            if (rank >= upto - mine && rank < upto) {
                while (left >= count[byte]) left -= count[byte++];
                rank_and_bits[0] = left;
                rank_and_bits[1] = known | byte << shift;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const bool any = nan_or_top[1] != 0, none = nan_or_top[0] && nan_or_top[1] < kInf;
        out[blockIdx.x].top = none ? __uint_as_float(0x7fc00000u) : __uint_as_float(nan_or_top[1]);
        out[blockIdx.x].low = none ? __uint_as_float(0x7fc00000u) : any ? __uint_as_float(rank_and_bits[1]) : 0.0f;
    }
}

void sizes_of(const SizeRuns& runs, Sizes* out, hipStream_t st) {
    hipLaunchKernelGGL(sizes_kernel, dim3(kSizeRuns), dim3(kSizesThreads), 0, st, runs, out);
    check(hipGetLastError(), "sizes_of");
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
