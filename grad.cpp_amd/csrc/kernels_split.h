// Projections over many rows on the bf16 matrix cores without losing fp32: every fp32
// operand is written as the sum of three bf16 numbers and the products of the parts are
// accumulated in fp32.
//
//   a = a1 + a2 + a3,  a1 = bf16(a), a2 = bf16(a - a1), a3 = bf16(a - a1 - a2)
//
// The split is exact in its range: rounding to nearest leaves |a - a1| <= 2^-9 |a| (16 significant bits),
// |a - a1 - a2| <= 2^-18 |a| (8 bits), which a3 holds whole.  A product of two such numbers
// needs the nine products of parts; the six kept here are those down to 2^-18 of a b
// (a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1).  The three left out sum to less than
// 2^-26 |a b|, an eighth of what rounding a b to fp32 loses (2^-24 |a b| / 2 each way), so an
// fp32 dot product formed this way is as good as one formed of fp32 products: both are
// dominated by the roundings of the running sum, and there are fewer of those here (one per
// 16 terms against one per 2).
//
// The range: from kSplitTop (3.396e38, the last 2^-9 below the largest float) a1 would be infinite
// and a2 not a number, so weights are checked when they are split, and a form with one that large,
// or an infinite one, is not used: its passes stay on fp32 products (a NaN is one either way).
// Activations are not checked; one there lies within 2^-9 of its own overflow.  Below 2^-103 the
// small parts are subnormal: at most 2^-125 times the other factor is lost, nothing in a sum that
// any ordinary weight takes part in.
//
// Why: on this part an fp32 matrix product runs at the vector rate (157 TFLOP/s; nothing
// vector issues beside it), a bf16 one at sixteen times that, so six of them are still 2.7
// times as fast.
#pragma once

#include "kernels_gemv.h"
#include "operand_format.h"

namespace gh {

// Rows of weights are stored in the order in which the accumulator hands outputs back: of
// every 32 outputs, lane half h of a 32 x 32 product holds matrix rows 8 q + 4 h + e (q, e in
// 0..3), and they are given to outputs 16 h + 4 q + e, so that a lane ends up with 16
// consecutive outputs of one row of activations.
__host__ __device__ __forceinline__ int split_output_of_row(int row) {
    const int rho = row & 31;
    return (row & ~31) + 16 * ((rho >> 2) & 1) + 4 * (rho >> 3) + (rho & 3);
}

// Writes the split form of a weight matrix src (N x K, row per output).  Row `row` of the split matrix is
// output split_output_of_row(row), zeros past N; *beyond is set if a weight is out of range.  gate_up: src rows are (gate, up) pairs, and
// every 16 outputs are the gates of eight hidden units and then their ups.
static __global__ __launch_bounds__(256) void split_weights_kernel(const float* __restrict__ src, int N, int K,
                                                                   int rows, int gate_up, char* dst, int* beyond) {
    const int chunks = K >> 3;
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= static_cast<size_t>(rows) * chunks) return;
    const int row = static_cast<int>(i / chunks), k = static_cast<int>(i % chunks) * 8;
    int n = split_output_of_row(row);
    if (gate_up) n = (n & ~15) + 2 * (n & 7) + ((n >> 3) & 1);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (n < N) {
        const float4 a = *reinterpret_cast<const float4*>(src + static_cast<size_t>(n) * K + k);
        const float4 b = *reinterpret_cast<const float4*>(src + static_cast<size_t>(n) * K + k + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    }
    bool out = false;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const unsigned size = __float_as_uint(v[e]) & 0x7FFFFFFFu;
        out |= size >= kSplitTop && size <= 0x7F800000u;
    }
    if (out) *beyond = 1;
    store_split8(dst, row, k, K / kSplitCols, v);
}

// norm(x) of a row (layer_norm_row, inference.cpp:30-58) by one wavefront; store(k, v) takes
// columns k .. k + 7.  The row stays in registers: NI chunks of eight columns per lane, d <= 512 NI.  Two chunks
// leave room for gamma, requested with the row instead of behind its sums (us per launch in pairs: RMS 1999 x 768
// 7.6 -> 6.5, 24576 x 768 36.0 -> 34.9, LayerNorm 16384 x 768 26.8 -> 25.8, with beta too 27.9; 2, 4 or 8 rows per workgroup
// are not faster).
template <bool RMS, int NI, class Store>
__device__ __forceinline__ void norm_row(const float* __restrict__ xr, const float* __restrict__ gamma,
                                         const float* __restrict__ beta, int d, int lane, Store store) {
    constexpr bool kEarly = NI <= 2;
    const int chunks = d >> 3;
    float v[NI][8], g[kEarly ? NI : 1][8];
    float s = 0.0f;
    if constexpr (kEarly) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int c = min(lane + 64 * i, chunks - 1);
#pragma unroll
            for (int e = 0; e < 8; e++) g[i][e] = gamma[c * 8 + e];
        }
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int c = lane + 64 * i;
        const bool in = c < chunks;
        const float4 a = in ? *reinterpret_cast<const float4*>(xr + c * 8) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 b = in ? *reinterpret_cast<const float4*>(xr + c * 8 + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[i][0] = a.x, v[i][1] = a.y, v[i][2] = a.z, v[i][3] = a.w;
        v[i][4] = b.x, v[i][5] = b.y, v[i][6] = b.z, v[i][7] = b.w;
        if (RMS) s += dot4(a, a) + dot4(b, b);
        else s += ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
    }
    s = wave_sum(s) / static_cast<float>(d);
    float scale;
    if (RMS) {
        scale = 1.0f / sqrtf(s + kNormEps);
    } else {
        float var = 0.0f;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            if (lane + 64 * i < chunks) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    v[i][e] -= s;
                    var += v[i][e] * v[i][e];
                }
            }
        }
        scale = 1.0f / sqrtf(wave_sum(var) / static_cast<float>(d) + kNormEps);
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int c = lane + 64 * i;
        if (c >= chunks) continue;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            o[e] = (kEarly ? g[kEarly ? i : 0][e] : gamma[c * 8 + e]) * v[i][e] * scale;
            if (!RMS) o[e] += beta[c * 8 + e];
        }
        store(c * 8, o);
    }
}

// The same for a row that does not fit the registers: one pass over it per sum and one to write,
// the later ones from the L2.
template <bool RMS, class Store>
__device__ __forceinline__ void norm_long_row(const float* __restrict__ xr, const float* __restrict__ gamma,
                                              const float* __restrict__ beta, int d, int lane, Store store) {
    float s = 0.0f;
    for (int k = lane * 4; k < d; k += 256) {
        const float4 a = *reinterpret_cast<const float4*>(xr + k);
        s += RMS ? dot4(a, a) : (a.x + a.y) + (a.z + a.w);
    }
    s = wave_sum(s) / static_cast<float>(d);
    const float mean = RMS ? 0.0f : s;
    if (!RMS) {
        s = 0.0f;
        for (int k = lane * 4; k < d; k += 256) {
            float4 a = *reinterpret_cast<const float4*>(xr + k);
            a = make_float4(a.x - mean, a.y - mean, a.z - mean, a.w - mean);
            s += dot4(a, a);
        }
        s = wave_sum(s) / static_cast<float>(d);
    }
    const float scale = 1.0f / sqrtf(s + kNormEps);
    for (int k = lane * 8; k < d; k += 512) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            o[e] = gamma[k + e] * (xr[k + e] - mean) * scale;
            if (!RMS) o[e] += beta[k + e];
        }
        store(k, o);
    }
}

// h = norm(x) of every row in split form, 16 rows per workgroup: it writes whole blocks.
template <bool RMS, int NI>
static __global__ __launch_bounds__(1024) void norm_split_kernel(const float* __restrict__ x,
                                                                 const float* __restrict__ gamma,
                                                                 const float* __restrict__ beta, char* out, int M,
                                                                 int d) {
    const int m = blockIdx.x * 16 + (threadIdx.x >> 6);
    if (m >= M) return;
    norm_row<RMS, NI>(x + static_cast<size_t>(m) * d, gamma, beta, d, threadIdx.x & 63,
                      [&](int k, const float(&o)[8]) { store_split8(out, m, k, d / kSplitCols, o); });
}

template <bool RMS>
static __global__ __launch_bounds__(1024) void norm_split_long_kernel(const float* __restrict__ x,
                                                                      const float* __restrict__ gamma,
                                                                      const float* __restrict__ beta, char* out, int M,
                                                                      int d) {
    const int m = blockIdx.x * 16 + (threadIdx.x >> 6);
    if (m >= M) return;
    norm_long_row<RMS>(x + static_cast<size_t>(m) * d, gamma, beta, d, threadIdx.x & 63,
                       [&](int k, const float(&o)[8]) { store_split8(out, m, k, d / kSplitCols, o); });
}

struct SplitGemmParams {
    const char* A;  // split activations, M rows (storage for whole tiles)
    const char* W;  // split weights (storage for whole tiles, outputs in split_output_of_row order)
    int M, N, K;
    int n_tiles, tiles;
    const float* bias;  // N floats or nullptr
    float* out;         // EPI_RESID: x.  EPI_QKV: q
    int out_stride;
    char* out_split;  // EPI_GELU, EPI_SWIGLU: split rows of out_cols columns
    int out_kblocks;
    // operands in pairs (kernels_pair.h)
    const float* unit;   // per output: what a sum's unit is worth, of W
    float operand_unit;  // ... of A
    float pair_scale;    // of the rows at out_split
    // EPI_QKV (rows of a prompt pass, as in GemvParams); outputs first .. first + N of the fused product
    int first;
    KvLayout kv;
    int layer, d_model, rope;
    const float *rope_cos, *rope_sin;
    int rows_per_seq, pos_base;
    // EPI_STORE: logits that are scored, not stored.  Every 64 outputs of a row leave
    // (largest, sum of exp(v - largest)), and the target's logit is kept.
    // Row m = seq * rows_per_seq + t is position nll_t0 + t of sequence seq.
    const int* targets;  // [batch][nll_len]
    int nll_t0, nll_len;
    float2* nll_part;  // [M][nll_stride]
    int nll_stride;    // n_tiles * WN
    float* nll_target;  // [M]
};

// Loads of 16 bytes per lane straight into LDS (lane i's bytes at lds + 16 i), counted by
// vmcnt.  Written as assembly because the compiler, which sees that such a load and an LDS
// read could meet, waits for every load in flight in front of each read; the waits that are
// needed are the ones split_gemm_kernel writes down.
__device__ __forceinline__ void load_to_lds(const char* base, unsigned lane_off, unsigned lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(base), "s"(lds)
                 : "memory");
}

template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Everything this wavefront has read from LDS is in registers, then the workgroup meets.
// (Not __syncthreads: that one waits for the loads in flight too.)
__device__ __forceinline__ void meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), in a form the compiler counts with
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The place of the tile-th tile: eight row tiles deep inside a column of outputs, so that what workgroups with
// neighbouring tiles read at about the same time is the same few tiles of both operands.
__device__ __forceinline__ void split_place(const SplitGemmParams& p, int tile, int& m_tile, int& n_tile) {
    const int m_tiles = p.tiles / p.n_tiles;
    const int group = tile / (8 * p.n_tiles), rest = tile - group * 8 * p.n_tiles;
    const int deep = min(8, m_tiles - group * 8);
    n_tile = rest / deep;
    m_tile = group * 8 + rest - n_tile * deep;
}

// The workgroup's tile.  Workgroup ids go round-robin over the eight XCDs: every XCD takes a contiguous run of
// tiles.  False: there is none for it.
__device__ __forceinline__ bool split_tile(const SplitGemmParams& p, int& m_tile, int& n_tile) {
    const int per = (p.tiles + 7) >> 3, id = blockIdx.x;
    const int tile = (id & 7) * per + (id >> 3);
    if ((id >> 3) >= per || tile >= p.tiles) return false;
    split_place(p, tile, m_tile, n_tile);
    return true;
}

// What the split projections make of their outputs, and how they leave rows of the next one's operand.
struct SplitRowsOut {
    static __device__ __forceinline__ float gelu(float x) { return gelu_tanh(x); }
    static __device__ __forceinline__ float silu(float x) { return gh::silu(x); }
    static __device__ __forceinline__ float exp_of(float x) { return expf(x); }
    static __device__ __forceinline__ void store8(const SplitGemmParams& p, int m, int k, const float (&v)[8]) {
        store_split8(p.out_split, m, k, p.out_kblocks, v);
    }
};

// What becomes of a wavefront's outputs, straight from the accumulators: register r of acc[a][b] is output
// n0 + 32 a + 16 (lane / 32) + r of row m0 + 32 b + lane % 32.  nll_at: the wavefront's run of outputs (EPI_STORE).
template <class Rows, int EPI, int MB, int NB>
__device__ __forceinline__ void split_epilogue(const SplitGemmParams& p, const v16f (&acc)[NB][MB], int m0, int n0, int nll_at) {
    const int lane = threadIdx.x & 63, r32 = lane & 31, h32 = lane >> 5;
#pragma unroll
    for (int b = 0; b < MB; b++) {
        const int m = m0 + 32 * b + r32;
        if constexpr (EPI == EPI_STORE) {
            // scored logits: no store, the row's running maximum and sum of exponentials
            float mx = -INFINITY;
            int target = -1;
            if (m < p.M) {
                const int seq = m / p.rows_per_seq, t = m - seq * p.rows_per_seq;
                target = p.targets[static_cast<size_t>(seq) * p.nll_len + p.nll_t0 + t];
            }
#pragma unroll
            for (int a = 0; a < NB; a++) {
                const int n = n0 + 32 * a + 16 * h32;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    if (n + r < p.N) mx = fmaxf(mx, acc[a][b][r]);
                    if (n + r == target) p.nll_target[m] = acc[a][b][r];
                }
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
            const float base = mx == -INFINITY ? 0.0f : mx;  // (nothing but -inf here: a mass of 0)
            float sum = 0.0f;
#pragma unroll
            for (int a = 0; a < NB; a++) {
                const int n = n0 + 32 * a + 16 * h32;
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (n + r < p.N) sum += Rows::exp_of(acc[a][b][r] - base);
            }
            sum += __shfl_xor(sum, 32, kWave);
            if (m < p.M && h32 == 0)
                p.nll_part[static_cast<size_t>(m) * p.nll_stride + nll_at] = make_float2(mx, sum);
        } else {
            if (m >= p.M) continue;
            int pos = 0, page = 0;
            if constexpr (EPI == EPI_QKV) {
                const int seq = m / p.rows_per_seq;
                pos = p.pos_base + (m - seq * p.rows_per_seq);
                page = p.kv.page_table[seq * p.kv.pages_per_seq + (pos >> p.kv.page_shift)];
            }
#pragma unroll
            for (int a = 0; a < NB; a++) {
                const int n = n0 + 32 * a + 16 * h32;
                if (n >= p.N) continue;
                float v[16];
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] = acc[a][b][r];
                if constexpr (EPI == EPI_RESID) {
                    // y += b, then y += x @ W (inference.cpp:22-28)
                    float4* out = reinterpret_cast<float4*>(p.out + static_cast<size_t>(m) * p.out_stride + n);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        float4 c = out[q];
                        if (p.bias) {
                            const float4 bb = *reinterpret_cast<const float4*>(p.bias + n + 4 * q);
                            c = make_float4(c.x + bb.x, c.y + bb.y, c.z + bb.z, c.w + bb.w);
                        }
                        out[q] = make_float4(c.x + v[4 * q], c.y + v[4 * q + 1], c.z + v[4 * q + 2], c.w + v[4 * q + 3]);
                    }
                } else if constexpr (EPI == EPI_GELU) {
                    float o[2][8];
#pragma unroll
                    for (int r = 0; r < 16; r++) o[r >> 3][r & 7] = Rows::gelu(v[r] + p.bias[n + r]);
                    Rows::store8(p, m, n, o[0]);
                    Rows::store8(p, m, n + 8, o[1]);
                } else if constexpr (EPI == EPI_SWIGLU) {
                    float o[8];
#pragma unroll
                    for (int r = 0; r < 8; r++) o[r] = v[8 + r] * Rows::silu(v[r]);
                    Rows::store8(p, m, n >> 1, o);
                } else if constexpr (EPI == EPI_QKV) {
                    const int sec = (p.first + n) / p.d_model, c = p.first + n - sec * p.d_model, head = c >> 6, j = c & 63;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4 bb = *reinterpret_cast<const float4*>(p.bias + p.first + n + 4 * q);
                        v[4 * q] += bb.x, v[4 * q + 1] += bb.y, v[4 * q + 2] += bb.z, v[4 * q + 3] += bb.w;
                    }
                    if (p.rope && sec < 2) {
                        const float* cs = p.rope_cos + pos * 32 + (j >> 1);
                        const float* sn = p.rope_sin + pos * 32 + (j >> 1);
#pragma unroll
                        for (int q = 0; q < 2; q++) {
                            const float4 c4 = *reinterpret_cast<const float4*>(cs + 4 * q);
                            const float4 s4 = *reinterpret_cast<const float4*>(sn + 4 * q);
                            const float cc[4] = {c4.x, c4.y, c4.z, c4.w}, ss[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const float x = v[8 * q + 2 * e], y = v[8 * q + 2 * e + 1];
                                v[8 * q + 2 * e] = x * cc[e] - y * ss[e];
                                v[8 * q + 2 * e + 1] = x * ss[e] + y * cc[e];
                            }
                        }
                    }
                    float* dst;
                    if (sec == 0) {
                        dst = p.out + static_cast<size_t>(m) * p.out_stride + c;
                    } else {
                        const size_t run = ((static_cast<size_t>(p.layer) * p.kv.n_pages + page) * 2 + (sec - 1)) * p.kv.heads + head;
                        dst = p.kv.pool + ((run << p.kv.page_shift) + (pos & ((1 << p.kv.page_shift) - 1))) * 64 + j;
                    }
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        reinterpret_cast<float4*>(dst)[q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
                }
            }
        }
    }
}

// C[M,N] = A[M,K] . W[N,K]^T, operands split.  A workgroup of WM x WN wavefronts owns
// 32 MB WM rows and 32 NB WN outputs, a wavefront 32 MB x 32 NB of them in accumulators of
// 32 x 32 (outputs along the matrix rows, so a lane holds one row of activations).  Operands
// pass through LDS in steps of 16 columns (one block), STAGES steps in the ring; a step's
// fragments are read from LDS under the products of the step before.  KG > 1: KG such
// sets of wavefronts, each with a ring of its own, share K and add up at the end.
template <int EPI, int MB, int NB, int WM, int WN, int KG, int STAGES, int PER_CU>
__global__ __launch_bounds__(64 * WM * WN * KG, PER_CU * WM * WN * KG / 4) void split_gemm_kernel(const SplitGemmParams p) {
    extern __shared__ __attribute__((aligned(1024))) char lds_split[];
    constexpr int kWaves = WM * WN, TM = 32 * MB * WM, TN = 32 * NB * WN;
    constexpr int kUnitsA = TM * kSplitRowBytes / 1024, kUnits = (TM + TN) * kSplitRowBytes / 1024;  // 1024-byte loads of a step
    constexpr int kLoads = (kUnits + kWaves - 1) / kWaves;  // ... per wavefront
    constexpr int kStage = kUnits * 1024;
    static_assert((KG - 1) * TM * TN * 4 <= KG * STAGES * kStage, "the sums fit in the rings");
    static_assert(kUnitsA * 1024 == TM * kSplitRowBytes && kUnits * 1024 == (TM + TN) * kSplitRowBytes, "whole loads");
    const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave_id / kWaves, wave = wave_id % kWaves;
    const int wm = wave / WN, wn = wave % WN;
    int m_tile, n_tile;
    if (!split_tile(p, m_tile, n_tile)) return;
    const int row_blocks = p.K / kSplitCols, kblocks = row_blocks / KG;  // of a row, of this set of wavefronts
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds_split))
                          + kg * (STAGES * kStage);
    // this wavefront's loads: units wave, wave + kWaves, ... of a step's image in LDS (the row
    // groups of A, then those of W, 1536 bytes each)
    const char* a_base = p.A + static_cast<size_t>(m_tile) * (TM / kSplitRows) * row_blocks * kSplitBlockBytes
                         + static_cast<size_t>(kg * kblocks) * kSplitBlockBytes;
    const char* w_base = p.W + static_cast<size_t>(n_tile) * (TN / kSplitRows) * row_blocks * kSplitBlockBytes
                         + static_cast<size_t>(kg * kblocks) * kSplitBlockBytes;
    unsigned src[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int u = min(wave + i * kWaves, kUnits - 1);  // (a load too many brings the last unit again)
        const unsigned at = (u < kUnitsA ? u : u - kUnitsA) * 1024 + lane * 16;
        const unsigned g = at / kSplitBlockBytes;
        src[i] = g * (row_blocks * kSplitBlockBytes) + (at - g * kSplitBlockBytes);
    }
    const auto issue_one = [&](int i, int step, int stage) {
        const int u = min(wave + i * kWaves, kUnits - 1);
        const char* at = (u < kUnitsA ? a_base : w_base) + static_cast<size_t>(step) * kSplitBlockBytes;
        load_to_lds(at, src[i], lds0 + stage * kStage + u * 1024);
    };
    // operand reads: row lane % 32 of a 32-row block, columns 8 (lane / 32) .. + 7
    const int r32 = lane & 31, h32 = lane >> 5;
    const int chunk_at = r32 * kSplitRowBytes + ((h32 ^ ((r32 >> 3) & 1)) << 4);
    // the parts of the rows of A and W of a step
    v8bf a0[MB], a1[MB], a2[MB], w0[NB], w1[NB], w2[NB];
    const auto read_a = [&](int stage, int q, v8bf (&f)[MB]) {
        const char* at = lds_split + (kg * STAGES + stage) * kStage + chunk_at + q * kSplitPartBytes;
#pragma unroll
        for (int x = 0; x < MB; x++) f[x] = *reinterpret_cast<const v8bf*>(at + (wm * MB + x) * 2 * kSplitBlockBytes);
    };
    const auto read_w = [&](int stage, int q, v8bf (&f)[NB]) {
        const char* at = lds_split + (kg * STAGES + stage) * kStage + chunk_at + q * kSplitPartBytes + TM / kSplitRows * kSplitBlockBytes;
#pragma unroll
        for (int x = 0; x < NB; x++) f[x] = *reinterpret_cast<const v8bf*>(at + (wn * NB + x) * 2 * kSplitBlockBytes);
    };
    // The products of the first parts and the other five in accumulators of their own: what
    // rounds in a sum of K products is the large running value, and the small products, added to
    // it one after the other, would round it five more times per 16 columns.
    v16f acc[NB][MB], low[NB][MB];
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = low[a][b][r] = 0.0f;
    const auto multiply = [&](const v8bf (&w)[NB], const v8bf (&x)[MB], v16f (&sum)[NB][MB]) {
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (int b = 0; b < MB; b++) sum[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[a], x[b], sum[a][b], 0, 0, 0);
    };

#pragma unroll
    for (int s = 0; s < STAGES; s++)
        if (s < kblocks) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) issue_one(i, s, s);
        }
    if (kblocks >= STAGES) wait_loads<(STAGES - 1) * kLoads>();
    else wait_loads<0>();
    meet();
    read_w(0, 0, w0);
    read_a(0, 2, a2);
    read_a(0, 1, a1);
    read_w(0, 1, w1);
    // A step's six rounds of products, in an order that uses up one part after the other, so
    // that a part of the next step is read into the registers of this step's a round or two
    // before it is needed (with every part in two places the 64 x 64 wavefronts run out of
    // registers).  Reads and loads go out between the rounds: all at once behind the meeting
    // they held up the first product of every wavefront.  One path through the loop: a second
    // copy of the products would hold the accumulators in other registers.
    int stage = 0;
    for (int s = 0; s < kblocks; s++) {
        const int next = stage == STAGES - 1 ? 0 : stage + 1;
        const bool more = s + STAGES < kblocks;
        const auto send = [&](int t) {  // a quarter of the loads of step s + STAGES, into this step's place
            constexpr int kPer = (kLoads + 3) / 4;
            if (more) {
#pragma unroll
                for (int i = t * kPer; i < (t + 1) * kPer; i++)
                    if (i < kLoads) issue_one(i, s + STAGES, stage);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        multiply(w0, a2, low);
        read_w(stage, 2, w2);
        __builtin_amdgcn_sched_barrier(0);
        multiply(w0, a1, low);
        read_a(stage, 0, a0);
        __builtin_amdgcn_sched_barrier(0);
        if (STAGES > 2 && s + STAGES <= kblocks) wait_loads<(STAGES - 2) * kLoads>();  // step s + 1 is here
        else wait_loads<0>();
        meet();  // ... for everyone, and everyone has read this step's place
        multiply(w0, a0, acc);
        read_a(next, 2, a2);
        send(0);
        multiply(w1, a1, low);
        read_w(next, 0, w0);
        send(1);
        multiply(w1, a0, low);
        read_a(next, 1, a1);
        send(2);
        multiply(w2, a0, low);
        read_w(next, 1, w1);
        send(3);
        stage = next;
    }
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[a][b] += low[a][b];
    if constexpr (KG > 1) {
        // the other sets' sums through the LDS the rings no longer need, added in order
        float* sums = reinterpret_cast<float*>(lds_split);
        const auto at = [&](int g, int a, int b) { return sums + (((g - 1) * kWaves + wave) * NB * MB + a * MB + b) * 1024 + lane; };
        __syncthreads();
        if (kg > 0) {
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = 0; b < MB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) at(kg, a, b)[r * 64] = acc[a][b][r];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int g = 1; g < KG; g++)
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = 0; b < MB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[a][b][r] += at(g, a, b)[r * 64];
    }

    split_epilogue<SplitRowsOut, EPI, MB, NB>(p, acc, m_tile * TM + wm * 32 * MB, n_tile * TN + wn * 32 * NB, n_tile * WN + wn);
}

// nll of a scored row from what the logits launch left of it: log of the sum of all
// exponentials, less the target's logit (Variable::cross_entropy, variable.cpp:589-592).  One
// wavefront per row; row seq * slice_len + t holds position t0 + t of sequence seq.
static __global__ __launch_bounds__(256) void nll_parts_kernel(const float2* __restrict__ part, int stride,
                                                               const float* __restrict__ target, int M, int slice_len,
                                                               int t0, int len, float* nll) {
    const int lane = threadIdx.x & 63, m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= M) return;
    const float2* row = part + static_cast<size_t>(m) * stride;
    float mx = -INFINITY;
    for (int i = lane; i < stride; i += 64) mx = fmaxf(mx, row[i].x);
    mx = wave_max(mx);
    float sum = 0.0f;
    for (int i = lane; i < stride; i += 64) {
        const float2 v = row[i];
        if (v.y != 0.0f) sum += v.y * expf(v.x - mx);  // (a run without mass has no maximum; NaN is mass)
    }
    sum = wave_sum(sum);
    if (lane == 0) {
        const int seq = m / slice_len, t = m - seq * slice_len;
        nll[static_cast<size_t>(seq) * len + t0 + t] = (logf(sum) + mx) - target[m];
    }
}

}  // namespace gh
