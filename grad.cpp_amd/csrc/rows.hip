// The many-row projections' variants and the rule that picks one, in a translation unit of
// their own.
#include "rows.h"

#include "kernels_pair_attn.h"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace gh {

static void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
}

void split_weights(const float* src, int N, int K, bool gate_up, char* dst, int* beyond, hipStream_t st) {
    const int rows = (N + kSplitPad - 1) / kSplitPad * kSplitPad;
    const size_t chunks = static_cast<size_t>(rows) * (K / 8);
    hipLaunchKernelGGL(split_weights_kernel, dim3(static_cast<unsigned>((chunks + 255) / 256)), dim3(256), 0, st, src, N,
                       K, rows, gate_up ? 1 : 0, dst, beyond);
    check(hipGetLastError(), "split_weights");
}

template <bool RMS>
static void norm_split_as(const float* x, const float* gamma, const float* beta, char* out, int M, int d, hipStream_t st) {
    const dim3 grid((M + 15) / 16), block(1024);
    if (d <= 1024) hipLaunchKernelGGL((norm_split_kernel<RMS, 2>), grid, block, 0, st, x, gamma, beta, out, M, d);
    else if (d <= 4096) hipLaunchKernelGGL((norm_split_kernel<RMS, 8>), grid, block, 0, st, x, gamma, beta, out, M, d);
    else hipLaunchKernelGGL((norm_split_long_kernel<RMS>), grid, block, 0, st, x, gamma, beta, out, M, d);
    check(hipGetLastError(), "norm_split");
}

void norm_split(bool rms, const float* x, const float* gamma, const float* beta, char* out, int M, int d, hipStream_t st) {
    if (rms) norm_split_as<true>(x, gamma, beta, out, M, d, st);
    else norm_split_as<false>(x, gamma, beta, out, M, d, st);
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
    switch (split_tiling(p.M, p.N, p.K)) {
        case SPLIT_32_K4: launch<EPI, 1, 1, 1, 1, 4, 3, 2>(p, st); break;
        case SPLIT_64_K4: launch<EPI, 1, 1, 2, 2, 4, 3, 1>(p, st); break;
        case SPLIT_64: launch<EPI, 1, 1, 2, 2, 1, 3, 4>(p, st); break;
        case SPLIT_128x64: launch<EPI, 2, 1, 2, 2, 1, 4, 2>(p, st); break;
        case SPLIT_128: launch<EPI, 2, 2, 2, 2, 1, 3, 2>(p, st); break;
    }
}

// Key tiles per workgroup, as a shift.  Query blocks are whole workgroups (128 queries against
// all their keys) while there are enough of them or the longest has six tiles at most (8
// sequences of 256 tokens: 18 us, shared 18 and 8 for the merge); below 640 workgroups the keys of the
// long blocks are shared, as coarsely as reaches 640 and so among 1300 or so at most (12 heads of 1999 tokens: 89 us unshared, 76 in runs of
// 1024 keys, 47 of 512, 46 of 256, 48 of 128; the merge cost 1, 6, 8, 12, 18 us more, that of
// 256 keys costs 9 since its loads go out together).
// attn_pair_kernel: 480 instead of 640 (12 heads of 1999 tokens with the merge: 44.6 us in runs of 256 keys, 42.3 of 512,
// 57.8 of 1024; 48 heads of 1024: 41.1 unshared, 39.9 of 512, 46.6 of 256).
static int attn_chunk_shift(int pairs, int len, int pos_base, bool in_pairs) {
    const int blocks = (len + kAttnQueries - 1) / kAttnQueries;
    int shift = 20;
    const auto workgroups = [&](int sh) {
        int n = 0;
        for (int i = 0; i < blocks; i++) n += attn_parts(i, len, pos_base, sh);
        return static_cast<long>(n) * pairs;
    };
    const int enough = in_pairs ? 480 : 640;
    if (workgroups(20) >= enough || attn_key_tiles(blocks - 1, len, pos_base) <= 6) return 20;
    for (shift = 14; shift > 1 && workgroups(shift) < enough; shift--) {
    }
    return shift;
}

static int attn_items(int len, int pos_base, int shift) {
    int n = 0;
    for (int i = 0; i * kAttnQueries < len; i++) n += attn_parts(i, len, pos_base, shift);
    return n;
}

// Pairs whose keys and values are split at a time.
static int attn_group(int pairs, int positions, size_t kv_bytes) {
    const size_t fit = kv_bytes / (static_cast<size_t>((positions + 63) / 64) * kAttnTile);
    return static_cast<int>(std::min<size_t>(std::max<size_t>(fit, 1), pairs));
}

// Splitting goes pair by pair anyway and a quarter of a gigabyte is thousands of workgroups' worth,
// so more would only be more memory.
size_t split_attention_kv_bytes(int batch, int heads, int positions) {
    const size_t pair = static_cast<size_t>((positions + 63) / 64) * kAttnTile;
    return std::max(pair, std::min(pair * batch * heads, size_t{256} << 20));
}

size_t split_attention_part_floats(int batch, int heads, int len, int pos_base, size_t kv_bytes, bool in_pairs) {
    size_t need = 0;
    const int pairs = batch * heads, group = attn_group(pairs, pos_base + len, kv_bytes);
    for (const int n : {group, pairs % group}) {
        const int shift = n ? attn_chunk_shift(n, len, pos_base, in_pairs) : 20;
        if (shift != 20) need = std::max(need, static_cast<size_t>(n) * attn_items(len, pos_base, shift) * kAttnPart);
    }
    return need;
}

void split_attention(const PrefillAttnParams& a, int batch, char* kv, size_t kv_bytes, float* part, hipStream_t st) {
    static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_split_kernel),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, kAttnLds);
    check(raised, "hipFuncSetAttribute");
    const bool in_pairs = a.pair_scale != 0.0f;
    const int heads = a.kv.heads, pairs = batch * heads, positions = a.pos_base + a.len;
    const int group = attn_group(pairs, positions, kv_bytes);
    const int blocks = (a.len + kAttnQueries - 1) / kAttnQueries;
    SplitAttnParams p{};
    p.q = a.q;
    p.kv = kv;
    p.tiles = (positions + 63) / 64;
    p.out = a.out_split;
    p.pair_scale = in_pairs ? 1.0f / kPairWeightScale : 0.0f;  // of merged parts (values carry that of the rows)
    p.key_unit = in_pairs ? 1.0f / a.key_scale : 0.0f;
    p.part = part;
    p.d_model = a.d_model;
    p.heads = heads;
    p.len = a.len;
    p.pos_base = a.pos_base;
    p.scale = a.scale;
    for (p.first = 0; p.first < pairs; p.first += group) {
        p.pairs = std::min(group, pairs - p.first);
        p.chunk_shift = attn_chunk_shift(p.pairs, a.len, a.pos_base, in_pairs);
        p.items = attn_items(a.len, a.pos_base, p.chunk_shift);
        const SplitKvParams k{a.kv, a.layer, p.first, positions, kv, a.key_scale, a.pair_scale};
        hipLaunchKernelGGL(in_pairs ? split_kv_kernel<2> : split_kv_kernel<3>, dim3(p.tiles, p.pairs), dim3(256), 0, st, k);
        check(hipGetLastError(), "split_kv");
        hipLaunchKernelGGL(in_pairs ? attn_pair_kernel : attn_split_kernel, dim3((p.pairs + 7) / 8 * 8 * p.items), dim3(256),
                           in_pairs ? kPairAttnLds : kAttnLds, st, p);
        check(hipGetLastError(), "attn_split");
        if (p.items > blocks) {
            hipLaunchKernelGGL(in_pairs ? attn_split_merge_kernel<true> : attn_split_merge_kernel<false>, dim3(4 * blocks, p.pairs), dim3(256), 0, st, p);
            check(hipGetLastError(), "attn_split_merge");
        }
    }
}

void nll_parts(const SplitGemmParams& p, float* nll, hipStream_t st) {
    hipLaunchKernelGGL(nll_parts_kernel, dim3((p.M + 3) / 4), dim3(256), 0, st, p.nll_part, p.nll_stride, p.nll_target,
                       p.M, p.rows_per_seq, p.nll_t0, p.nll_len, nll);
    check(hipGetLastError(), "nll_parts");
}

template void split_gemm<EPI_STORE>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_QKV>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_RESID>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_GELU>(SplitGemmParams&, hipStream_t);
template void split_gemm<EPI_SWIGLU>(SplitGemmParams&, hipStream_t);

}  // namespace gh
