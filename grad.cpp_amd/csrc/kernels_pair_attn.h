// Causal attention of a prompt pass on the fp16 matrix cores, operands in two parts like those of the projections
// (kernels_pair.h): three products for one fp32 product, head size 64.
#pragma once

#include "kernels_split_attn.h"

namespace gh {

// Tiles of 64 positions as split_kv_kernel<2> leaves them: K, 64 rows (keys) x 64 columns, then V^T as four steps of 16
// keys, each 64 rows (dims) x 16 columns; second parts 2^11 larger.
constexpr int kPairAttnOperand = 16 * kPairBlockBytes;
constexpr int kPairAttnTile = 2 * kPairAttnOperand;
constexpr int kPairAttnRing = 4;
constexpr int kPairAttnLds = kPairAttnRing * kPairAttnOperand;
constexpr float kPairWeightScale = 16384.0f;  // of the probabilities: fp16's upper end

// attn_split_kernel's work and order: 128 queries per workgroup against a run of key tiles, both products transposed.
// What differs:
// - A query is scaled by a power of two of its own, from its largest element, and its scores come back with it (in the
//   multiply-add that takes off the maximum).  Probabilities are split 2^14 larger; values carry the power of
//   two of the rows that leave.
// - Of a tile's twelve products per 32 x 32 block the eight small ones go first, over all of K = 64, then the four of the first
//   parts: four roundings of a full-sized sum, where three parts had 24.  (Sums of 64 terms against float64, over the
//   size of the result: 0.98e-7 with the small products apart, 1.09e-7 with the six of three parts in turn.)
// - The workgroup meets once per tile, its ring four operands deep, and a product's fragments are all read well ahead: values
//   in front of the softmax, the next keys behind the products with them.  The softmax takes one kind of step over all 32 scores
//   after the other (pair by pair each step waited for the one before).
// 16 x 12 heads, us, three parts -> two in that kernel's form -> as it is: 1024 tokens 206 -> 110 -> 106, 1536 400 -> 221 -> 215;
// 1 x 12 x 1999 48 -> 36 -> 34 (the first with each form's best order of workgroups).  What bounds it: 48 products and 290 vector
// instructions per wavefront and tile, two wavefronts per SIMD.  The next tile's scores formed beside the softmax, a product
// every 8, 12 or 16 instructions: 7 % slower; a ring of five, one of them a tile further ahead: no faster.
static __global__ __launch_bounds__(256, 2) void attn_pair_kernel(const SplitAttnParams p) {
    extern __shared__ __attribute__((aligned(1024))) char lds_pair_attn[];
    int pair, b, h, item;
    if (!attn_place(p, pair, b, h, item)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n32 = lane & 31, h32 = lane >> 5;
    // longest query blocks first
    int qb = (p.len + kAttnQueries - 1) / kAttnQueries - 1, chunk = item, parts;
    while (chunk >= (parts = attn_parts(qb, p.len, p.pos_base, p.chunk_shift))) {
        chunk -= parts;
        qb--;
    }
    const int tile0 = chunk << p.chunk_shift;
    const int tile1 = min(tile0 + (1 << p.chunk_shift), attn_key_tiles(qb, p.len, p.pos_base));
    const int t = qb * kAttnQueries + wave * 32 + n32;  // this lane's query (token index in the pass)
    const int qpos = p.pos_base + min(t, p.len - 1);
    const int wave_last = p.pos_base + min(p.len, qb * kAttnQueries + wave * 32 + 32) - 1;  // last key of this wavefront
    const int wave_first = p.pos_base + min(p.len - 1, qb * kAttnQueries + wave * 32);      // position of its first query

    const char* const src = p.kv + static_cast<size_t>(pair) * p.tiles * kPairAttnTile;
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds_pair_attn));
    constexpr int kLoads = kPairAttnOperand / 1024 / 4;  // per wavefront and operand: one in front of each step
    const int operands = 2 * (tile1 - tile0);
    // load i of operand j: K (even) or V^T (odd) of tile tile0 + j / 2
    const auto issue = [&](int j, int i) {
        const char* at = src + static_cast<size_t>(2 * tile0 + j) * kPairAttnOperand;
        load_to_lds(at, (wave * kLoads + i) * 1024 + lane * 16,
                    lds0 + (j & (kPairAttnRing - 1)) * kPairAttnOperand + (wave * kLoads + i) * 1024);
    };
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < kLoads; i++) issue(min(j, operands - 1), i);

    // Q^T: dims 16 c + 8 (lane / 32) .. + 7 of the lane's query, in units of ln 2
    v8h q1[4], q2[4];
    float unit;  // of the lane's scores
    {
        const float qscale = p.scale * 1.44269504088896341f;
        const float* qr = p.q + (static_cast<size_t>(b) * p.len + min(t, p.len - 1)) * p.d_model + h * 64;
        float v[4][8], top = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float4 x = *reinterpret_cast<const float4*>(qr + c * 16 + h32 * 8);
            const float4 y = *reinterpret_cast<const float4*>(qr + c * 16 + h32 * 8 + 4);
            v[c][0] = x.x * qscale, v[c][1] = x.y * qscale, v[c][2] = x.z * qscale, v[c][3] = x.w * qscale;
            v[c][4] = y.x * qscale, v[c][5] = y.y * qscale, v[c][6] = y.z * qscale, v[c][7] = y.w * qscale;
#pragma unroll
            for (int i = 0; i < 8; i++) top = fmaxf(top, fabsf(v[c][i]));
        }
        top = fmaxf(top, __shfl_xor(top, 32, kWave));
        // the largest goes to [2^14, 2^15), a query below 2^-112, or one near that against small keys, stays lower: its unit has to
        // be a number other than zero, or a masked score were none (and its scores differ by less than 2^-60)
        const int s = top > 0.0f && top < INFINITY ? min(14 - ilogbf(top), 126 + min(ilogbf(p.key_unit), 0)) : 0;
        const float up = ldexpf(1.0f, s);
        unit = ldexpf(p.key_unit, -s);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            v4u a, b;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                unsigned first, second;
                to_pairs(v[c][2 * i] * up, v[c][2 * i + 1] * up, 1.0f, first, second);
                a[i] = first, b[i] = second;
            }
            q1[c] = __builtin_bit_cast(v8h, a);
            q2[c] = __builtin_bit_cast(v8h, b);
        }
    }
    const _Float16 down = static_cast<_Float16>(1.0f / kPairLift);
    v16f o[2], zero;  // O^T: dims 32 db + 8 (r / 4) + 4 (lane / 32) + r % 4 of the lane's query
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.0f;
    o[0] = o[1] = zero;
    float m = -INFINITY, l = 0.0f;

    const int row_at = (n32 & 15) * 16 + h32 * kPairChunkBytes;
    const int k_at = (n32 >> 4) * 4 * kPairBlockBytes + row_at, v_at = (n32 >> 4) * kPairBlockBytes + row_at;
    const auto place = [&](int j) { return lds_pair_attn + (j & (kPairAttnRing - 1)) * kPairAttnOperand; };
    // A tile's product: fragments of its four steps of two 32-row blocks, read all at once and well ahead.
    v8h f1[4][2], f2[4][2];
    const auto fetch = [&](const char* at, int step, int far) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                f2[c][i] = *reinterpret_cast<const v8h*>(at + c * step + i * far + kPairPartBytes);
                f1[c][i] = *reinterpret_cast<const v8h*>(at + c * step + i * far);
            }
    };
    const auto fetch_keys = [&](int j) { fetch(place(j) + k_at, kPairBlockBytes, 8 * kPairBlockBytes); };
    const auto fetch_values = [&](int j) { fetch(place(j) + v_at, 4 * kPairBlockBytes, 2 * kPairBlockBytes); };
    const auto product = [&](const v8h (&g1)[4], const v8h (&g2)[4], v16f (&out)[2]) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const v8h low = g1[c] * down;
#pragma unroll
            for (int i = 0; i < 2; i++)
                out[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f2[c][i], low, c == 0 ? zero : out[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; i++) out[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[c][i], g2[c], out[i], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 2; i++) out[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[c][i], g1[c], out[i], 0, 0, 0);
    };

    wait_loads<2 * kLoads>();  // the first tile's keys
    meet();
    fetch_keys(0);
    for (int kt = tile0; kt < tile1; kt++) {
        const int j = 2 * (kt - tile0), kh = kt * 64;
        const bool future = kh > wave_last;  // every key of the tile lies behind this wavefront's queries
        v16f sc[2];
        if (!future) product(q1, q2, sc);
        // this tile's values and the next one's keys are here, and everyone is done with the operands before them
        wait_loads<0>();
        meet();
        if (j + 3 < operands) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) issue(j + 3, i);
            if (j + 4 < operands) {
#pragma unroll
                for (int i = 0; i < kLoads; i++) issue(j + 4, i);
            }
        }
        if (future) continue;
        fetch_values(j + 1);
        __builtin_amdgcn_sched_barrier(0);
        // causal mask (keys up to the query's own position)
        if (kh + 63 > wave_first) {  // only the tiles on the diagonal need the comparisons
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = kh + kb * 32 + 8 * (r >> 2) + 4 * h32 + (r & 3);
                    sc[kb][r] = (key <= qpos) ? sc[kb][r] : -INFINITY;
                }
        }
        float mb = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) mb = fmaxf(mb, sc[kb][r]);
        mb = fmaxf(mb, __shfl_xor(mb, 32, kWave)) * unit;  // the two halves of a wavefront hold different keys of a query
        const float mn = fmaxf(m, mb);
        const float base = mn == -INFINITY ? 0.0f : mn;   // (a query may have no key in this run of tiles yet)
        const float f = __builtin_amdgcn_exp2f(m - base);  // 0 on the first tile
        // (one kind of step over all of them after the other: pair by pair every step waits for the one before)
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) sc[kb][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][r], unit, -base));
        __builtin_amdgcn_sched_barrier(0);
        float sums[4] = {0.f, 0.f, 0.f, 0.f};
        v8h p1[4], p2[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            v4u a, b;
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                x[i] = sc[s >> 1][(s & 1) * 8 + i];
                sums[i & 3] += x[i];
                x[i] *= kPairWeightScale;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                unsigned first, second;
                to_pairs(x[2 * i], x[2 * i + 1], 1.0f, first, second);
                a[i] = first, b[i] = second;
            }
            p1[s] = __builtin_bit_cast(v8h, a);
            p2[s] = __builtin_bit_cast(v8h, b);
        }
        float psum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
        psum += __shfl_xor(psum, 32, kWave);
        l = l * f + psum;
        m = mn;
        v16f tile[2];
        product(p1, p2, tile);
        fetch_keys(j + 2);  // (past the last tile: of whatever lies there, not used)
#pragma unroll
        for (int db = 0; db < 2; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[db][r] = o[db][r] * f + tile[db][r];
    }
    if (parts > 1) {
        float* part = p.part + (static_cast<size_t>(pair) * p.items + item) * kAttnPart + wave * (34 * 64) + lane;
        part[0] = m;
        part[64] = l;
#pragma unroll
        for (int r = 0; r < 32; r++) part[(2 + r) * 64] = o[r >> 4][r & 15];
        return;
    }
    if (t >= p.len) return;
    const float inv = 1.0f / (l * kPairWeightScale);
#pragma unroll
    for (int db = 0; db < 2; db++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++)
            store_pair4(p.out, b * p.len + t, h * 64 + db * 32 + q4 * 8 + h32 * 4, p.d_model / kSplitCols, o[db][4 * q4] * inv,
                        o[db][4 * q4 + 1] * inv, o[db][4 * q4 + 2] * inv, o[db][4 * q4 + 3] * inv, 1.0f);
}

}  // namespace gh
