// Projections over many rows on the fp16 matrix cores: every fp32 operand as the sum of two fp16
// numbers, three products of parts for one fp32 product.
//
//   a 2^s = a1 + a2,  a1 = fp16(a 2^s), a2 = fp16(a 2^s - a1)
//
// (Two half-precision parts, the second lifted by 2^11 and the sums taken out of the matrix core against its truncation: as
// published by Ootomo and Yokota, 2022.)
//
// What that costs and what pays for it.  a1 + a2 holds 22 bits and a sign, so a value is at most one unit
// of its 24th bit away (a quarter of all values are; half a unit rms, where rounding to fp32 leaves 0.29),
// and a2 b2 (2^-22 of the product at most) is left out: 7.5e-8 of a dot product's size, whatever its length.
// The six products of the exact three-part form (kernels_split.h) lose nothing there, but their sums are K / 16 terms
// added one after the other, and those roundings grow with K.  Here every 64 columns are summed from zero and
// then added to the running sum: 4 (or 12, see pair_tile) and K / 64 roundings.  The matrix cores cut the low bits of what they
// align, downwards: a bias of 2e-8 (K = 768) to 4e-8 (2048) of the result, the same in every row, which an attention over
// many positions would not average out; so the weights of every other 64 columns are stored negated and their
// sums subtracted (what is left is below 1e-9).  Error over the size of the result against float64, normal operands, three
// parts with K in one set / in four -> two: K = 512 1.28 / 0.77e-7 -> 1.09 to 1.26, 768 1.59 / 0.88 -> 1.12 to 1.32, 1024
// 1.86 / 0.98 -> 1.14 to 1.37, 2048 2.72 / 1.34 -> 1.19 to 1.27, 3072 3.40 / 1.63 -> 1.25 to 1.38 (the upper end 128 x 128
// and 128 x 64 tiles; an fp32 sum of one product after the other: 4.0 to 9.9).  Few rows whose products four sets would
// share take three parts (parts_are_closer in tilings.h).  Below K = 512 the three parts are the closer ones, so narrower
// models keep them (kPairMinCols).
//
// The range.  fp16 has exponents -14 to 15 and, below, numbers of fewer bits (the matrix cores take them as
// they are).  Weights are scaled row by row so that a row's largest lies in [2^14, 2^15).  Activations have one power of two
// per operand, from a bound that holds for every input (pair_bounds in engine.hip): nothing can
// overflow, and how far a bound lies above what occurs costs nothing: a2 of an activation is
// stored 2^11 larger, and meets a1 of the weight 2^-11 smaller, so that an activation keeps its 22 bits down to
// 2^-29 of the bound, and a weight down to 2^-17 of its row's largest; what is smaller is off by 2^-51 of the
// bound, or 2^-40 of the row's largest.  Models whose bounds lie further above what occurs than that leaves room
// for keep the three parts.
//
// Why: a third fewer bytes per operand and half the products.  In turn on one box, 128 x 128 tiles, operands of
// full-length significands: 16384 x 768 x 3072 180 -> 342 TFLOP/s of fp32 products, 24576 x 4096 x 768 180 -> 277,
// 1999 x 768 x 2048 136 -> 198 (best tile of either).
#pragma once

#include "epilogue_math.h"
#include "kernels_split.h"

namespace gh {

constexpr int kPairStages = 4;  // of the ring of steps; also the steps of a part

// Sign that the weights of block `block` of a row are stored with.
__host__ __device__ __forceinline__ float pair_sign(int block) { return (block & kPairStages) ? -1.0f : 1.0f; }

// Writes the pairs of a weight matrix src (N x K, row per output), rows in the order of split_weights_kernel, one
// wavefront per row, zeros past N.  unit[j]: the power of two that output j's sum is to be multiplied by, j as the
// product counts them; norm[n]: the 2-norm of row n of src, infinite if the row has no pairs: a weight is 2^40 or more
// (units stay far inside fp32), or more than an eighth of them (zeros aside) lie 2^14 and more below the largest.
static __global__ __launch_bounds__(256) void pair_weights_kernel(const float* __restrict__ src, int N, int K, int rows,
                                                                  int gate_up, char* dst, float* unit, float* norm) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int out = split_output_of_row(row);  // as the product hands it back
    const int n = gate_up ? (out & ~15) + 2 * (out & 7) + ((out >> 3) & 1) : out;
    const float* const w = src + static_cast<size_t>(min(n, N - 1)) * K;
    float top = 0.0f;
    for (int k = lane * 4; k < K; k += 256) {
        const float4 a = *reinterpret_cast<const float4*>(w + k);
        top = fmaxf(fmaxf(top, fmaxf(fabsf(a.x), fabsf(a.y))), fmaxf(fabsf(a.z), fabsf(a.w)));
    }
    top = wave_max(top);
    // the largest goes to [2^14, 2^15); a row below 2^-40 stays lower, and is off by 2^-79 at most
    const int s = top > 0.0f && top < INFINITY ? min(14 - ilogbf(top), 54) : 0;
    const float scale = ldexpf(1.0f, s), high = ldexpf(top, s - 14);
    float sum = 0.0f, some = 0.0f, most = 0.0f;  // weights that are not zero, and those within 2^14 of the largest
    for (int k = lane * 4; k < K; k += 256) {
        const float4 a = *reinterpret_cast<const float4*>(w + k);
        const float v[4] = {a.x * scale, a.y * scale, a.z * scale, a.w * scale};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sum += v[i] * v[i];
            some += v[i] != 0.0f ? 1.0f : 0.0f;
            most += fabsf(v[i]) >= high ? 1.0f : 0.0f;
        }
    }
    sum = wave_sum(sum);
    const bool fit = top < 0x1p40f && wave_sum(most) * 8.0f >= wave_sum(some) * 7.0f;
    if (lane == 0) unit[out] = out < N ? ldexpf(1.0f, -s) : 0.0f;
    if (lane == 0 && n < N) norm[n] = fit ? ldexpf(sqrtf(sum), -s) : INFINITY;
    for (int k = lane * 8; k < K; k += 512) {
        const float factor = scale * pair_sign(k >> 4);
        v4u p1, p2;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float x = w[k + 2 * i], y = w[k + 2 * i + 1];
            unsigned a, b;
            to_pairs(n < N ? x * factor : 0.0f, n < N ? y * factor : 0.0f, 1.0f, a, b);
            p1[i] = a;
            p2[i] = b;
        }
        char* at = dst + pair_offset(row, k, K >> 4);
        *reinterpret_cast<v4u*>(at) = p1;
        *reinterpret_cast<v4u*>(at + kPairPartBytes) = p2;
    }
}

// norm(x) of every row as pairs: norm_split_kernel with its sums, and its rows in registers.
template <bool RMS, int NI>
static __global__ __launch_bounds__(1024) void norm_pair_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                                const float* __restrict__ beta, char* out, int M, int d,
                                                                float pair_scale) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 16 + (threadIdx.x >> 6);
    if (m >= M) return;
    norm_row<RMS, NI>(x + static_cast<size_t>(m) * d, gamma, beta, d, lane,
                      [&](int k, const float(&o)[8]) { store_pair8(out, m, k, d / kSplitCols, o, pair_scale); });
}

template <bool RMS>
static __global__ __launch_bounds__(1024) void norm_pair_long_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                                     const float* __restrict__ beta, char* out, int M, int d,
                                                                     float pair_scale) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 16 + (threadIdx.x >> 6);
    if (m >= M) return;
    norm_long_row<RMS>(x + static_cast<size_t>(m) * d, gamma, beta, d, lane,
                       [&](int k, const float(&o)[8]) { store_pair8(out, m, k, d / kSplitCols, o, pair_scale); });
}

// The epilogues' functions: figures in epilogue_math.h.
struct DeviceUnit {
    static __device__ __forceinline__ float exp2(float x) { return __builtin_amdgcn_exp2f(x); }
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
};

struct PairRowsOut : EpilogueMath<DeviceUnit> {
    static __device__ __forceinline__ void store8(const SplitGemmParams& p, int m, int k, const float (&v)[8]) {
        store_pair8(p.out_split, m, k, p.out_kblocks, v, p.pair_scale);
    }
};

// EPI_RESID and EPI_QKV leave in strips of 8 rows x 32 outputs (lane / 8 the row, four outputs per lane), after a turn of
// a 32 x 32 block through LDS.  A lane of the accumulators holds 16 outputs of one row: from there an instruction
// touched 64 lines for 16 bytes each, a strip is eight whole lines.  What a strip reads, of memory that nobody else writes
// meanwhile, is requested in front of the products.  Where sets share K, all of them add and store strips,
// instead of the first set alone.  Same sums in the same order.  us per launch, before -> after: W_o and FFN2 of 16384
// rows 159 -> 155 (a GPT of 768 columns), of 24576 191 -> 176 (a Llama of 768), QKV 197 -> 181 and 287 -> 267, 2048 rows' W_o and FFN2 23.0 -> 21.5;
// over 160 to 16384 rows 4 to 11 % less.  A residual's bias and units held the same way from the start were slower (128 x 128:
// 253 registers, 0.995 of before instead of 0.945); QKV's are held where the wavefront's sums are its own (0.95 -> 0.91).
constexpr int kTurnStride = 36, kTurnFloats = 32 * kTurnStride;  // of a block of 32 x 32

__device__ __forceinline__ void turn_block(float* lds, const v16f& v) {
    const int lane = threadIdx.x & 63;
    float* const to = lds + (lane & 31) * kTurnStride + 16 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; q++) *reinterpret_cast<float4*>(to + 4 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
}

__device__ __forceinline__ float4 turned_strip(const float* lds, int i) {
    const int lane = threadIdx.x & 63;
    return *reinterpret_cast<const float4*>(lds + (8 * i + (lane >> 3)) * kTurnStride + (lane & 7) * 4);
}

struct StripRow {  // EPI_QKV
    int pos, page;
};

struct StripColumns {  // EPI_QKV: of the lane's four outputs
    float4 unit, bias;
};

__device__ __forceinline__ StripColumns strip_columns(const SplitGemmParams& p, int n) {
    // (storage of units for whole tiles, as of the weights)
    return {*reinterpret_cast<const float4*>(p.unit + n),
            n < p.N ? *reinterpret_cast<const float4*>(p.bias + p.first + n) : make_float4(0.f, 0.f, 0.f, 0.f)};
}

__device__ __forceinline__ StripRow strip_row(const SplitGemmParams& p, int m) {
    const int row = min(m, p.M - 1), seq = row / p.rows_per_seq, pos = p.pos_base + (row - seq * p.rows_per_seq);
    return {pos, p.kv.page_table[seq * p.kv.pages_per_seq + (pos >> p.kv.page_shift)]};
}

__device__ __forceinline__ float4 strip_operand(const SplitGemmParams& p, int m, int n) {  // EPI_RESID
    return m < p.M && n < p.N ? *reinterpret_cast<const float4*>(p.out + static_cast<size_t>(m) * p.out_stride + n)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
}

// Outputs n .. n + 3 of row m.
__device__ __forceinline__ void strip_resid(const SplitGemmParams& p, int m, int n, const float4& y, const float4& v) {
    // y += b, then y += x @ W (inference.cpp:22-28)
    float4 c = y;
    if (p.bias) {
        const float4 bb = *reinterpret_cast<const float4*>(p.bias + n);
        c = make_float4(c.x + bb.x, c.y + bb.y, c.z + bb.z, c.w + bb.w);
    }
    *reinterpret_cast<float4*>(p.out + static_cast<size_t>(m) * p.out_stride + n) = make_float4(c.x + v.x, c.y + v.y, c.z + v.z, c.w + v.w);
}

__device__ __forceinline__ void strip_qkv(const SplitGemmParams& p, int m, int n, const StripRow& r, const float4& bb, const float4& v) {
    const int of = p.first + n, sec = (of >= p.d_model) + (of >= 2 * p.d_model), c = of - sec * p.d_model, j = c & 63;
    float4 o = make_float4(v.x + bb.x, v.y + bb.y, v.z + bb.z, v.w + bb.w);
    if (p.rope && sec < 2) {
        const float2 cs = *reinterpret_cast<const float2*>(p.rope_cos + r.pos * 32 + (j >> 1));
        const float2 sn = *reinterpret_cast<const float2*>(p.rope_sin + r.pos * 32 + (j >> 1));
        o = make_float4(o.x * cs.x - o.y * sn.x, o.x * sn.x + o.y * cs.x, o.z * cs.y - o.w * sn.y, o.z * sn.y + o.w * cs.y);
    }
    float* dst;
    if (sec == 0) {
        dst = p.out + static_cast<size_t>(m) * p.out_stride + c;
    } else {
        const size_t run = ((static_cast<size_t>(p.layer) * p.kv.n_pages + r.page) * 2 + (sec - 1)) * p.kv.heads + (c >> 6);
        dst = p.kv.pool + ((run << p.kv.page_shift) + (r.pos & ((1 << p.kv.page_shift) - 1))) * 64 + j;
    }
    *reinterpret_cast<float4*>(dst) = o;
}

// C[M,N] = A[M,K] . W[N,K]^T of pairs.  Tiles, workgroup order, LDS ring and epilogues are split_gemm_kernel's. A step
// of 16 columns is three rounds of products (w1 a2, w2 a1, w1 a1), its fragments read from LDS during the step before
// into registers of their own (a 64 x 64 wavefront has 128 of its 256 for sums).  Four steps make a 64-column part that
// starts from zero and is then added to the running sums (or taken from them, the weights of every other part being
// negative).  (Added in front of the next part's products instead, accumulator by accumulator, the compiler copies every
// part first.)  In wavefronts of 32 rows the small products of a part (those with a second part) have a sum of their
// own: a full-sized sum is then cut four times a part instead of twelve (error of K = 512 1.26 -> 1.09e-7, 768 1.32 ->
// 1.12, 2048 1.55 -> 1.20 to 1.27, 3072 1.71 -> 1.25 to 1.38; 2000 rows of 768 columns 21.2 -> 21.8 us by its 16
// additions per block and part).  Those of 64 rows, which take the larger passes, are the closer ones without it and pay
// more for it (128 x 64 tiles, 8192 rows of W_o and FFN2 61.6 -> 68.5 us; 64 x 64 wavefronts have no registers left).  K
// / KG is a multiple of 64.
template <int EPI, int MB, int NB, int WM, int WN, int KG>
__device__ __forceinline__ void pair_tile(const SplitGemmParams& p, int m_tile, int n_tile) {
    extern __shared__ __attribute__((aligned(1024))) char lds_pair[];
    constexpr int kWaves = WM * WN, TM = 32 * MB * WM, TN = 32 * NB * WN, kStages = kPairStages;
    constexpr int kUnitsA = TM / 16, kUnits = (TM + TN) / 16;  // 1024-byte loads of a step: a block each
    constexpr int kLoads = (kUnits + kWaves - 1) / kWaves;     // ... per wavefront
    constexpr int kStage = kUnits * 1024;
    static_assert((KG - 1) * TM * TN * 4 <= KG * kStages * kStage, "the sums fit in the rings");
    const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave_id / kWaves, wave = wave_id % kWaves;
    const int wm = wave / WN, wn = wave % WN;
    const int row_blocks = p.K / kSplitCols, kblocks = row_blocks / KG;  // of a row, of this set of wavefronts
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds_pair))
                          + kg * (kStages * kStage);
    const char* a_base = p.A + (static_cast<size_t>(m_tile) * kUnitsA * row_blocks + kg * kblocks) * kPairBlockBytes;
    const char* w_base = p.W + (static_cast<size_t>(n_tile) * (kUnits - kUnitsA) * row_blocks + kg * kblocks) * kPairBlockBytes;
    // this wavefront's loads: units wave, wave + kWaves, ... of a step's image in LDS (the row groups of A, then those of W)
    unsigned src[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int u = min(wave + i * kWaves, kUnits - 1);  // (a load too many brings the last unit again)
        src[i] = (u < kUnitsA ? u : u - kUnitsA) * (row_blocks * kPairBlockBytes) + lane * 16;
    }
    const auto issue_one = [&](int i, int step, int stage) {
        const int u = min(wave + i * kWaves, kUnits - 1);
        const char* at = (u < kUnitsA ? a_base : w_base) + static_cast<size_t>(step) * kPairBlockBytes;
        load_to_lds(at, src[i], lds0 + stage * kStage + u * 1024);
    };
    // operand reads: row lane % 32 of a 32-row block, columns 8 (lane / 32) .. + 7
    const int r32 = lane & 31, h32 = lane >> 5;
    const char* const frag = lds_pair + kg * (kStages * kStage) + (r32 >> 4) * kPairBlockBytes + h32 * kPairChunkBytes + (r32 & 15) * 16;
    v8h a1[2][MB], a2[2][MB], w1[2][NB], w2[2][NB];  // fragments of even and odd steps
    const auto read_a = [&](int stage, int part, v8h (&f)[MB]) {
#pragma unroll
        for (int x = 0; x < MB; x++)
            f[x] = *reinterpret_cast<const v8h*>(frag + stage * kStage + part * kPairPartBytes + (wm * MB + x) * 2 * kPairBlockBytes);
    };
    const auto read_w = [&](int stage, int part, v8h (&f)[NB]) {
#pragma unroll
        for (int x = 0; x < NB; x++)
            f[x] = *reinterpret_cast<const v8h*>(frag + stage * kStage + part * kPairPartBytes
                                                 + (kUnitsA + (wn * NB + x) * 2) * kPairBlockBytes);
    };
    constexpr bool kApart = MB == 1;  // small products in sums of their own
    v16f sum[NB][MB], part[NB][MB], small[kApart ? NB : 1][kApart ? MB : 1], zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.0f;
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++) sum[a][b] = zero;
    const auto multiply = [&](const v8h (&w)[NB], const v8h (&x)[MB], auto& to, bool first) {
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (int b = 0; b < MB; b++) to[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[a], x[b], first ? zero : to[a][b], 0, 0, 0);
    };
    // Strips: of the wavefront's own blocks, or, where sets share K, every kAll-th of the tile's.
    // (QKV's 64 x 96 tiles with K shared by two sets are as fast without: 700 x 1920 x 640 13.9 us against 14.0, 700 and 1000 x 3072 x
    // 1024 24.9 and 29.3 against 25.1 and 29.4.)
    constexpr bool kStrips = EPI == EPI_RESID || (EPI == EPI_QKV && !(NB == 3 && KG == 2));
    constexpr int kAll = kWaves * KG, kCount = KG == 1 ? MB * NB * 4 : TM * TN / 256 / kAll;
    static_assert(!kStrips || kCount * 256 * kAll == TM * TN, "whole rounds of strips");
    const int col = (lane & 7) * 4;
    const auto strip_block = [&](int i) { return KG == 1 ? i >> 2 : (wave_id + i * kAll) >> 2; };  // a * MB + b; of the tile: row by row
    const auto strip_at = [&](int i) { return KG == 1 ? i & 3 : (wave_id + i * kAll) & 3; };
    const auto strip_m = [&](int i) {
        const int block = strip_block(i);
        return m_tile * TM + (KG == 1 ? (wm * MB + block % MB) * 32 : block / (TN / 32) * 32) + strip_at(i) * 8 + (lane >> 3);
    };
    const auto strip_n = [&](int i) {
        const int block = strip_block(i);
        return n_tile * TN + (KG == 1 ? (wn * NB + block / MB) * 32 : block % (TN / 32) * 32) + col;
    };
    constexpr bool kColumnsEarly = EPI == EPI_QKV && KG == 1;
    StripColumns cols[kColumnsEarly ? NB : 1];
    if constexpr (kColumnsEarly) {
#pragma unroll
        for (int a = 0; a < NB; a++) cols[a] = strip_columns(p, strip_n(a * MB * 4));
    }
    float4 y[EPI == EPI_RESID ? kCount : 1];
    StripRow row[EPI == EPI_QKV && kStrips ? (KG == 1 ? MB * 4 : kCount) : 1];
    if constexpr (EPI == EPI_RESID) {
#pragma unroll
        for (int i = 0; i < kCount; i++) y[i] = strip_operand(p, strip_m(i), strip_n(i));
    }
    if constexpr (EPI == EPI_QKV && kStrips) {
#pragma unroll
        for (int i = 0; i < (KG == 1 ? MB * 4 : kCount); i++) row[i] = strip_row(p, strip_m(i));
    }
#pragma unroll
    for (int s = 0; s < kStages; s++)
#pragma unroll
        for (int i = 0; i < kLoads; i++) issue_one(i, s, s);
    wait_loads<(kStages - 1) * kLoads>();
    meet();
    read_w(0, 0, w1[0]);
    read_a(0, 1, a2[0]);
    read_w(0, 1, w2[0]);
    read_a(0, 0, a1[0]);
    for (int s0 = 0; s0 < kblocks; s0 += kStages) {
#pragma unroll
        for (int t = 0; t < kStages; t++) {  // step s0 + t, in place t of the ring
            constexpr int kPer = (kLoads + 2) / 3;
            const int c = t & 1, n = c ^ 1, next = (t + 1) % kStages;
            const bool more = s0 + t + kStages < kblocks;
            const auto send = [&](int q) {  // a third of the loads of the step that comes to this place next
                if (more) {
#pragma unroll
                    for (int i = q * kPer; i < (q + 1) * kPer; i++)
                        if (i < kLoads) issue_one(i, s0 + t + kStages, t);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            if (s0 + t + kStages - 1 < kblocks) wait_loads<(kStages - 2) * kLoads>();  // the next step is here
            else wait_loads<0>();
            meet();  // ... for everyone, and everyone has read this step's place
            v8h low[NB];
#pragma unroll
            for (int a = 0; a < NB; a++) low[a] = w1[c][a] * static_cast<_Float16>(1.0f / kPairLift);
            if constexpr (kApart) multiply(low, a2[c], small, t == 0);
            else multiply(low, a2[c], part, t == 0);
            read_w(next, 0, w1[n]);
            read_a(next, 1, a2[n]);
            send(0);
            if constexpr (kApart) multiply(w2[c], a1[c], small, false);
            else multiply(w2[c], a1[c], part, false);
            read_w(next, 1, w2[n]);
            send(1);
            multiply(w1[c], a1[c], part, kApart && t == 0);
            read_a(next, 0, a1[n]);
            send(2);
        }
        const float sign = pair_sign(kg * kblocks + s0);
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (int b = 0; b < MB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float v = part[a][b][r];
                    if constexpr (kApart) v += small[a][b][r];
                    sum[a][b][r] = __builtin_fmaf(v, sign, sum[a][b][r]);
                }
    }
    const auto scaled = [&](const float4& v, const float4& unit) {
        const float f = p.operand_unit;
        return make_float4(v.x * (unit.x * f), v.y * (unit.y * f), v.z * (unit.z * f), v.w * (unit.w * f));
    };
    const auto strip_out = [&](int i, const float4& v) {
        const int m = strip_m(i), n = strip_n(i);
        if (m >= p.M || n >= p.N) return;
        if constexpr (EPI == EPI_RESID) {
            strip_resid(p, m, n, y[i], v);
        } else if constexpr (kColumnsEarly) {
            const StripColumns& c = cols[i / (MB * 4)];
            strip_qkv(p, m, n, row[i % (MB * 4)], c.bias, scaled(v, c.unit));
        } else if constexpr (EPI == EPI_QKV) {
            strip_qkv(p, m, n, row[i], *reinterpret_cast<const float4*>(p.bias + p.first + n), v);
        }
    };
    if constexpr (KG > 1 && kStrips) {
        // Every set leaves its sums in the LDS that the rings no longer need; a strip's are added in the sets' order.
        constexpr int kBlocks = TM * TN / 1024;
        static_assert(KG * kBlocks * kTurnFloats * 4 <= KG * kStages * kStage, "they fit in the rings");
        float* const sums = reinterpret_cast<float*>(lds_pair);
        __syncthreads();
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (int b = 0; b < MB; b++)
                turn_block(sums + (kg * kBlocks + (wm * MB + b) * (TN / 32) + wn * NB + a) * kTurnFloats, sum[a][b]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kCount; i++) {
            float4 v = turned_strip(sums + strip_block(i) * kTurnFloats, strip_at(i));
#pragma unroll
            for (int g = 1; g < KG; g++) {
                const float4 w = turned_strip(sums + (g * kBlocks + strip_block(i)) * kTurnFloats, strip_at(i));
                v = make_float4(v.x + w.x, v.y + w.y, v.z + w.z, v.w + w.w);
            }
            strip_out(i, scaled(v, *reinterpret_cast<const float4*>(p.unit + strip_n(i))));
        }
        return;
    }
    if constexpr (KG > 1) {
        // the other sets' sums through the LDS the rings no longer need, added in order
        float* sums = reinterpret_cast<float*>(lds_pair);
        const auto at = [&](int g, int a, int b) { return sums + (((g - 1) * kWaves + wave) * NB * MB + a * MB + b) * 1024 + lane; };
        __syncthreads();
        if (kg > 0) {
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = 0; b < MB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) at(kg, a, b)[r * 64] = sum[a][b][r];
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
                    for (int r = 0; r < 16; r++) sum[a][b][r] += at(g, a, b)[r * 64];
    }
    const int n0 = n_tile * TN + wn * 32 * NB;
    if constexpr (!kColumnsEarly) {
#pragma unroll
        for (int a = 0; a < NB; a++) {
            // (storage of units for whole tiles, as of the weights)
            const float4* const u = reinterpret_cast<const float4*>(p.unit + n0 + 32 * a + 16 * h32);
            float units[16];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 v = u[q];
                units[4 * q] = v.x, units[4 * q + 1] = v.y, units[4 * q + 2] = v.z, units[4 * q + 3] = v.w;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float f = units[r] * p.operand_unit;
#pragma unroll
                for (int b = 0; b < MB; b++) sum[a][b][r] *= f;
            }
        }
    }
    if constexpr (kStrips) {
        // (every wavefront has its last step's fragments, so the rings' places are free, one block's to each)
        static_assert(kWaves * kTurnFloats * 4 <= kStages * kStage, "they fit in the ring");
        float* const block = reinterpret_cast<float*>(lds_pair) + wave * kTurnFloats;
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (int b = 0; b < MB; b++) {
                turn_block(block, sum[a][b]);
#pragma unroll
                for (int i = 0; i < 4; i++) strip_out((a * MB + b) * 4 + i, turned_strip(block, i));
            }
    } else {
        split_epilogue<PairRowsOut, EPI, MB, NB>(p, sum, m_tile * TM + wm * 32 * MB, n0, n_tile * WN + wn);
    }
}

template <int EPI, int MB, int NB, int WM, int WN, int KG, int PER_CU>
__global__ __launch_bounds__(64 * WM * WN * KG, PER_CU * WM * WN * KG / 4) void pair_gemm_kernel(const SplitGemmParams p) {
    int m_tile, n_tile;
    if (split_tile(p, m_tile, n_tile)) pair_tile<EPI, MB, NB, WM, WN, KG>(p, m_tile, n_tile);
}

// Tiles of 128 x 128, those behind the first `whole` (whole rounds of 256 compute units) in quarters of 64 x 64, dealt
// over the XCDs the same way; sums are those of either tiling.  Its time is one whole tile's chain of steps and epilogue
// with a quarter beside it: the matrix cores' share is a quarter of it (2000 x 2304 x 768).  Figures and the line at
// pair_tiling.
template <int EPI>
__global__ __launch_bounds__(256, 2) void pair_mixed_kernel(const SplitGemmParams p, int whole) {
    const int id = blockIdx.x;
    int m_tile, n_tile;
    if (id < whole) {
        split_place(p, (id & 7) * (whole >> 3) + (id >> 3), m_tile, n_tile);
        pair_tile<EPI, 2, 2, 2, 2, 1>(p, m_tile, n_tile);
    } else {
        const int per = (p.tiles - whole + 7) >> 3, slot = (id - whole) >> 3, quarter = slot & 3;
        const int tile = whole + (id & 7) * per + (slot >> 2);
        if ((slot >> 2) >= per || tile >= p.tiles) return;
        split_place(p, tile, m_tile, n_tile);
        m_tile = 2 * m_tile + (quarter >> 1);
        n_tile = 2 * n_tile + (quarter & 1);
        if (m_tile * 64 < p.M && n_tile * 64 < p.N) pair_tile<EPI, 1, 1, 2, 2, 1>(p, m_tile, n_tile);
    }
}

}  // namespace gh
