// Host side of the many-row projections (kernels_split.h).
#pragma once

#include "kernels_attn.h"
#include "kernels_split.h"
#include "tilings.h"

namespace gh {

constexpr int kSplitPad = 128;  // rows of a split matrix are allocated in whole tiles of this many

inline size_t split_bytes(size_t rows, size_t cols) {
    return (rows + kSplitPad - 1) / kSplitPad * kSplitPad * cols * 6;
}

// Writes the split form of src (N x K); gate_up: src rows are (gate, up) pairs.  *beyond is set if
// a weight is outside the range of the parts.
void split_weights(const float* src, int N, int K, bool gate_up, char* dst, int* beyond, hipStream_t st);

// norm(x) of M rows in split form.
void norm_split(bool rms, const float* x, const float* gamma, const float* beta, char* out, int M, int d, hipStream_t st);

// One projection; p.n_tiles, p.tiles (and p.nll_stride) are filled in.  EPI_STORE: scoring.
template <int EPI>
void split_gemm(SplitGemmParams& p, hipStream_t st);

// The same three in pairs; units of a matrix: one per row of its storage.
// (whole tiles of 96 outputs, also from a row behind the first)
inline size_t pair_rows(size_t rows) { return (rows + 95 + kSplitPad - 1) / kSplitPad * kSplitPad; }
inline size_t pair_bytes(size_t rows, size_t cols) { return pair_rows(rows) * cols * 4; }
void pair_weights(const float* src, int N, int K, bool gate_up, char* dst, float* unit, float* norm, hipStream_t st);
// Sizes of runs of values, of which the bounds of operands in pairs are made: the largest magnitude, and one that seven of eight
// of those that are not zero reach (a mean would follow the largest); not numbers where one of the values is none and the
// largest is finite.
struct Sizes {
    float top, low;
};
constexpr int kSizeRuns = 16;
struct SizeRuns {
    const float* at[kSizeRuns];
    int n[kSizeRuns];  // 0: no values, sizes of 0
};
void sizes_of(const SizeRuns& runs, Sizes* out, hipStream_t st);  // kSizeRuns of them
void norm_pair(bool rms, const float* x, const float* gamma, const float* beta, char* out, int M, int d, float pair_scale,
               hipStream_t st);
template <int EPI>
void pair_gemm(SplitGemmParams& p, hipStream_t st);

// Causal attention of p.len new positions of every sequence over the cache, output rows in split form.
// kv: scratch of kv_bytes, at least one (sequence, head) pair's keys and values; the pairs go in groups
// that fit.  split_attention_kv_bytes: what is worth giving for so many filled positions.
// part: scratch of the size split_attention_part_floats names for the call.
size_t split_attention_kv_bytes(int batch, int heads, int positions);
size_t split_attention_part_floats(int batch, int heads, int len, int pos_base, size_t kv_bytes, bool in_pairs);
void split_attention(const PrefillAttnParams& p, int batch, char* kv, size_t kv_bytes, float* part, hipStream_t st);

// Widest run of partial results per row that split_gemm<EPI_STORE> leaves.
inline int split_nll_stride(int N) { return (N + kSplitPad - 1) / kSplitPad * 4; }

// nll of M scored rows from those partial results.
void nll_parts(const SplitGemmParams& p, float* nll, hipStream_t st);

}  // namespace gh
