// Causal attention of a prompt pass on the bf16 matrix cores, operands split like those of the
// projections (kernels_split.h): six bf16 products for one fp32 product, head size 64.
#pragma once

#include "kernels_split.h"

namespace gh {

// K and V of the layer at hand in split form, for the length of one attention launch: per
// (sequence, head) tiles of 64 positions, 48 KB each: K as a split matrix of 64 rows (keys) x 64 columns (dims),
// then V^T as four steps of 16 keys, each a split matrix of 64 rows (dims) x 16 columns.
// Inside a step the keys come in the order 0-3, 8-11, 4-7, 12-15: what a lane half of the
// score product holds in consecutive registers (below).
constexpr int kAttnOperand = 64 * 4 * kSplitRowBytes;  // 24 KB
constexpr int kAttnTile = 2 * kAttnOperand;

// A launch covers a run of the (sequence, head) pairs, sequence by sequence.
struct SplitKvParams {
    KvLayout kv;
    int layer;
    int first;      // pair of workgroups y = 0
    int positions;  // filled positions of every sequence
    char* out;      // [pairs of the launch][ceil(positions / 64)][kAttnTile]
    float key_scale, value_scale;  // in two parts (kernels_pair_attn.h): their powers of two
};

// One workgroup per tile; rows past the last position become zeros (their scores are masked,
// and a weight of zero times what an earlier pass left must stay zero).
// PARTS: 3, or 2 in the same order (tiles of 32 KB).
template <int PARTS>
static __global__ __launch_bounds__(256) void split_kv_kernel(const SplitKvParams p) {
    constexpr int kOperand = PARTS == 3 ? kAttnOperand : 64 * 4 * kPairBlockBytes / 16;
    constexpr int kStep = PARTS == 3 ? 4 * kSplitBlockBytes : 4 * kPairBlockBytes;  // 16 keys of V^T
    const auto store = [](char* at, int row, int k, int kblocks, const float(&v)[8], float scale) {
        if constexpr (PARTS == 3) store_split8(at, row, k, kblocks, v);
        else store_pair8(at, row, k, kblocks, v, scale);
    };
    __shared__ float vs[64][65];
    const int tile = blockIdx.x, tid = threadIdx.x;
    const int pair = p.first + blockIdx.y, b = pair / p.kv.heads, h = pair - b * p.kv.heads;
    char* out = p.out + (static_cast<size_t>(blockIdx.y) * gridDim.x + tile) * (2 * kOperand);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = (tid >> 3) + 32 * i, k = (tid & 7) * 8, pos = tile * 64 + row;
        float kx[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float4 va = make_float4(0.f, 0.f, 0.f, 0.f), vb = va;
        if (pos < p.positions) {
            const float* kr = p.kv.pool + kv_offset(p.kv, p.layer, b, 0, h, pos) + k;
            const float* vr = kr + (static_cast<size_t>(p.kv.heads) << p.kv.page_shift) * 64;
            const float4 ka = *reinterpret_cast<const float4*>(kr), kb = *reinterpret_cast<const float4*>(kr + 4);
            kx[0] = ka.x, kx[1] = ka.y, kx[2] = ka.z, kx[3] = ka.w, kx[4] = kb.x, kx[5] = kb.y, kx[6] = kb.z, kx[7] = kb.w;
            va = *reinterpret_cast<const float4*>(vr);
            vb = *reinterpret_cast<const float4*>(vr + 4);
        }
        store(out, row, k, 4, kx, p.key_scale);
        vs[row][k] = va.x, vs[row][k + 1] = va.y, vs[row][k + 2] = va.z, vs[row][k + 3] = va.w;
        vs[row][k + 4] = vb.x, vs[row][k + 5] = vb.y, vs[row][k + 6] = vb.z, vs[row][k + 7] = vb.w;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int u = tid + 256 * i, c = u & 1, dim = (u >> 1) & 63, s = u >> 7;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = vs[16 * s + 4 * c + (j & 3) + 8 * (j >> 2)][dim];
        store(out + kOperand + s * kStep, dim, 8 * c, 1, v, p.value_scale);
    }
}

struct SplitAttnParams {
    const float* q;  // [batch * len][d_model], rotated
    const char* kv;  // split_kv_kernel's tiles
    int tiles;       // ... per pair
    char* out;       // operand rows [batch * len] x d_model
    float pair_scale;  // ... of pairs
    float* part;     // partial results of query blocks whose keys are shared among workgroups
    int d_model, heads, len, pos_base;
    int chunk_shift;  // a workgroup takes up to 1 << chunk_shift tiles of keys
    int items;        // workgroups per pair
    int first, pairs;  // the pairs of this launch
    float scale;
    float key_unit;  // in two parts: what a key's unit is worth, a power of two
};

// Workgroup ids go round-robin over the eight XCDs.  With many (sequence, head) pairs all workgroups of one sit on one
// XCD (192 pairs, three parts, pair by pair: 1024 tokens 247 -> 198 us, 1536 tokens 411 -> 388); with few the pairs
// would not spread evenly (12 pairs, 1999 tokens: 47 -> 57 us) and ids are dealt as they come.  On an XCD the longest
// query blocks of up to kAttnGroup pairs go first, then the next longest: pair by pair, a last pair's longest block
// began when the others were nearly done (192 pairs, attn_pair_kernel: 1024 tokens 140 -> 106 us, 1536 264 -> 220),
// which counts for more than an L2 of 4 MB that holds four pairs' tiles instead of 24.  us in groups of 4 / 12 / 24 / 48
// / 96: 96 pairs x 1024 61 / 55 / 55 / 55 / 55, 192 x 2000 411 / 384 / 384 / 385 / 385, 384 x 1000 219 / 215 / 212 / 212
// / 212, 768 x 500 133 / 135 / 131 / 135 / 137, 768 x 256 48 / 47 / 45 / 46 / 48. pair: counted from the launch's first.
// False for an id past the last pair.
constexpr int kAttnGroup = 24;

__device__ __forceinline__ bool attn_place(const SplitAttnParams& p, int& pair, int& b, int& h, int& item) {
    const int id = static_cast<int>(blockIdx.x);
    if (p.pairs >= 64 || (p.pairs & 7) == 0) {
        const int mine = (p.pairs + 7) >> 3, slot = id >> 3, g = slot / (kAttnGroup * p.items);
        const int rest = slot - g * kAttnGroup * p.items, deep = min(kAttnGroup, mine - g * kAttnGroup);
        item = rest / deep;
        pair = (id & 7) + 8 * (g * kAttnGroup + rest - item * deep);
    } else {
        pair = id / p.items;
        item = id - pair * p.items;
    }
    b = (p.first + pair) / p.heads;
    h = p.first + pair - b * p.heads;
    return pair < p.pairs;
}

constexpr int kAttnQueries = 128;
constexpr int kAttnRing = 3;
constexpr int kAttnLds = kAttnRing * kAttnOperand;
constexpr int kAttnPart = 4 * 34 * 64;  // floats of one partial result: [wavefront][m, l, o][lane]

// Tiles of keys in front of query block i, and the workgroups that share them.
__host__ __device__ __forceinline__ int attn_key_tiles(int i, int len, int pos_base) {
    const int end = (i + 1) * kAttnQueries;
    return (pos_base + (end < len ? end : len) + 63) >> 6;
}
__host__ __device__ __forceinline__ int attn_parts(int i, int len, int pos_base, int chunk_shift) {
    return (attn_key_tiles(i, len, pos_base) + (1 << chunk_shift) - 1) >> chunk_shift;
}

// One workgroup = 128 consecutive queries of one (sequence, head), 32 per wavefront, against a
// run of key tiles.  Both products are formed transposed,
//   S^T[key][query] = K . Q^T : a lane holds one query (lane % 32) and, of every block of 32 keys,
//   keys 8 (r / 4) + 4 (lane / 32) + r % 4 for r = 0..15,
// and a step of 16 keys of O^T[dim][query] += V^T . P^T takes registers 8 s .. 8 s + 7 of a block as
// they lie, V^T's columns being stored in that order.  The online softmax is
// inference.cpp:211-225 a tile at a time, in units of ln 2 (the scale carries log2 e, the
// exponential is the hardware's 2^x).  A tile's products go into accumulators that start at
// zero and are added to the running output once, the small products first: fewer roundings
// than one per product of two terms.
// K and V^T tiles arrive by loads straight into LDS, a ring of three operands: one being
// multiplied, one landed or landing, one on its way; two workgroups per compute unit, so
// that one's softmax (about 380 vector instructions per wavefront and tile, 170 of them the
// split of the probabilities) runs beside the other's 96 products.
static __global__ __launch_bounds__(256, 2) void attn_split_kernel(const SplitAttnParams p) {
    extern __shared__ __attribute__((aligned(1024))) char lds_attn[];
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

    const char* const src = p.kv + static_cast<size_t>(pair) * p.tiles * kAttnTile;
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds_attn));
    constexpr int kLoads = kAttnOperand / 1024 / 4;  // per wavefront and operand: two in front of each of three steps
    const int operands = 2 * (tile1 - tile0);
    // loads first .. last - 1 of operand j: K (even) or V^T (odd) of tile tile0 + j / 2
    const auto issue = [&](int j, int slot, int first, int last) {
        const char* at = src + static_cast<size_t>(2 * tile0 + j) * kAttnOperand;
#pragma unroll
        for (int i = first; i < last; i++)
            load_to_lds(at, (wave * kLoads + i) * 1024 + lane * 16, lds0 + slot * kAttnOperand + (wave * kLoads + i) * 1024);
    };
    issue(0, 0, 0, kLoads);
    issue(1, 1, 0, kLoads);

    // Q^T, split: dims 16 c + 8 (lane / 32) .. + 7 of the lane's query
    v8bf qf[4][3];
    {
        const float qscale = p.scale * 1.44269504088896341f;
        const float* qr = p.q + (static_cast<size_t>(b) * p.len + min(t, p.len - 1)) * p.d_model + h * 64;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float4 x = *reinterpret_cast<const float4*>(qr + c * 16 + h32 * 8);
            const float4 y = *reinterpret_cast<const float4*>(qr + c * 16 + h32 * 8 + 4);
            const float v[8] = {x.x * qscale, x.y * qscale, x.z * qscale, x.w * qscale,
                                y.x * qscale, y.y * qscale, y.z * qscale, y.w * qscale};
            v4u w[3];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                unsigned p1, p2, p3;
                split_pair(v[2 * i], v[2 * i + 1], p1, p2, p3);
                w[0][i] = p1, w[1][i] = p2, w[2][i] = p3;
            }
#pragma unroll
            for (int q = 0; q < 3; q++) qf[c][q] = __builtin_bit_cast(v8bf, w[q]);
        }
    }
    v16f o[2];  // O^T: dims 32 db + 8 (r / 4) + 4 (lane / 32) + r % 4 of the lane's query
#pragma unroll
    for (int db = 0; db < 2; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;

    const int row_at = (n32 & 15) * kSplitRowBytes + ((h32 ^ ((n32 >> 3) & 1)) << 4);
    const int k_at = (n32 >> 4) * 4 * kSplitBlockBytes + row_at, v_at = (n32 >> 4) * kSplitBlockBytes + row_at;
    // fragments of two 32-row blocks, `far` bytes apart
    const auto read = [&](const char* at, int far, v8bf (&f)[2][3]) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int q = 0; q < 3; q++) f[i][q] = *reinterpret_cast<const v8bf*>(at + i * far + q * kSplitPartBytes);
    };
    const auto multiply = [&](const v8bf (&f)[2][3], const v8bf (&g)[3], v16f (&sum)[2]) {
        constexpr int kFirst[6] = {2, 0, 1, 1, 0, 0}, kSecond[6] = {0, 2, 1, 0, 1, 0};  // small products first
#pragma unroll
        for (int x = 0; x < 6; x++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                sum[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i][kFirst[x]], g[kSecond[x]], sum[i], 0, 0, 0);
    };

    int slot = 0;  // of the operand being multiplied
    const auto arrive = [&](int j) {  // operand j has landed everywhere, and everyone is done with operand j - 1
        if (j + 1 < operands) wait_loads<kLoads>();
        else wait_loads<0>();
        meet();
    };
    const auto send = [&](int j, int first, int last) {  // operand j + 2 sets out, to the place of operand j - 1
        if (j + 2 < operands) issue(j + 2, slot == 0 ? 2 : slot - 1, first, last);
    };
    for (int kt = tile0; kt < tile1; kt++) {
        const int j = 2 * (kt - tile0), kh = kt * 64;
        const bool future = kh > wave_last;  // every key of the tile lies behind this wavefront's queries
        arrive(j);
        v8bf pf[4][3];
        float f = 1.0f;
        if (!future) {
            const char* at = lds_attn + slot * kAttnOperand + k_at;
            v16f sc[2];
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 16; r++) sc[kb][r] = 0.0f;
            v8bf fr[2][2][3];
            read(at, 8 * kSplitBlockBytes, fr[0]);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (c < 3) read(at + (c + 1) * kSplitBlockBytes, 8 * kSplitBlockBytes, fr[(c + 1) & 1]);
                if (c < 3) send(j, 2 * c, 2 * c + 2);
                __builtin_amdgcn_sched_barrier(0);  // the reads and loads go out before the products
                multiply(fr[c & 1], qf[c], sc);
            }
            // causal mask (keys up to the query's own position) and the tile's maximum per query
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
            mb = fmaxf(mb, __shfl_xor(mb, 32, kWave));  // the two halves of a wavefront hold different keys of a query
            const float mn = fmaxf(m, mb);
            const float base = mn == -INFINITY ? 0.0f : mn;  // (a query may have no key in this run of tiles yet)
            f = __builtin_amdgcn_exp2f(m - base);            // 0 on the first tile
            float psum = 0.0f;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                v4u w[3];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = __builtin_amdgcn_exp2f(sc[s >> 1][(s & 1) * 8 + 2 * i] - base);
                    const float y = __builtin_amdgcn_exp2f(sc[s >> 1][(s & 1) * 8 + 2 * i + 1] - base);
                    psum += x + y;
                    unsigned p1, p2, p3;
                    split_pair(x, y, p1, p2, p3);
                    w[0][i] = p1, w[1][i] = p2, w[2][i] = p3;
                }
#pragma unroll
                for (int q = 0; q < 3; q++) pf[s][q] = __builtin_bit_cast(v8bf, w[q]);
            }
            psum += __shfl_xor(psum, 32, kWave);
            l = l * f + psum;
            m = mn;
        } else {
            send(j, 0, kLoads);
        }
        slot = slot == kAttnRing - 1 ? 0 : slot + 1;
        arrive(j + 1);
        if (!future) {
            const char* at = lds_attn + slot * kAttnOperand + v_at;
            v16f tile[2];
#pragma unroll
            for (int db = 0; db < 2; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) tile[db][r] = 0.0f;
            v8bf fr[2][2][3];
            read(at, 2 * kSplitBlockBytes, fr[0]);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (s < 3) read(at + (s + 1) * 4 * kSplitBlockBytes, 2 * kSplitBlockBytes, fr[(s + 1) & 1]);
                if (s < 3) send(j + 1, 2 * s, 2 * s + 2);
                __builtin_amdgcn_sched_barrier(0);
                multiply(fr[s & 1], pf[s], tile);
            }
#pragma unroll
            for (int db = 0; db < 2; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[db][r] = o[db][r] * f + tile[db][r];
        } else {
            send(j + 1, 0, kLoads);
        }
        slot = slot == kAttnRing - 1 ? 0 : slot + 1;
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
    const float inv = 1.0f / l;
#pragma unroll
    for (int db = 0; db < 2; db++)
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++)
            store_split4(p.out, b * p.len + t, h * 64 + db * 32 + q4 * 8 + h32 * 4, p.d_model / kSplitCols, o[db][4 * q4] * inv,
                         o[db][4 * q4 + 1] * inv, o[db][4 * q4 + 2] * inv, o[db][4 * q4 + 3] * inv);
}

// Folds the partial results of a query block, in the order of the keys.  A chain of trips to memory, one per
// part (a part's rows were written by another workgroup): so a workgroup takes 32 queries only and a wavefront 8 of
// their 32 registers, and kMergeAhead parts are requested together.  12 heads x 1999 queries in up to 8 parts: 12.7 us ->
// 9.3 (4 TB/s), against four times the queries per workgroup, 32 registers per wavefront and a part at a time.
constexpr int kMergeAhead = 4;

template <bool PAIRS>
static __global__ __launch_bounds__(256) void attn_split_merge_kernel(const SplitAttnParams p) {
    const int pair = p.first + blockIdx.y, b = pair / p.heads, h = pair - b * p.heads;
    const int lane = threadIdx.x & 63, h32 = lane >> 5;
    const int r0 = (threadIdx.x >> 6) * 8, rows = blockIdx.x & 3;  // this wavefront's registers, the workgroup's 32 queries
    const int qb = (p.len + kAttnQueries - 1) / kAttnQueries - 1 - static_cast<int>(blockIdx.x >> 2);
    int first = 0;
    for (int i = qb + 1; i * kAttnQueries < p.len; i++) first += attn_parts(i, p.len, p.pos_base, p.chunk_shift);
    const int parts = attn_parts(qb, p.len, p.pos_base, p.chunk_shift), t = qb * kAttnQueries + rows * 32 + (lane & 31);
    if (parts == 1 || t >= p.len) return;
    const float* part = p.part + (static_cast<size_t>(blockIdx.y) * p.items + first) * kAttnPart + rows * (34 * 64) + lane;
    const auto at = [&](int c) { return part + static_cast<size_t>(min(c, parts - 1)) * kAttnPart; };
    float m = -INFINITY, l = 0.0f, o[8];
    for (int c = 0; c < parts; c += 2 * kMergeAhead) {
        float v[2 * kMergeAhead];
#pragma unroll
        for (int i = 0; i < 2 * kMergeAhead; i++) v[i] = at(c + i)[0];
#pragma unroll
        for (int i = 0; i < 2 * kMergeAhead; i++) m = fmaxf(m, v[i]);
    }
#pragma unroll
    for (int r = 0; r < 8; r++) o[r] = 0.0f;
    for (int c = 0; c < parts; c += kMergeAhead) {
        float v[kMergeAhead][10];
#pragma unroll
        for (int i = 0; i < kMergeAhead; i++) {
            v[i][8] = at(c + i)[0];
            v[i][9] = at(c + i)[64];
#pragma unroll
            for (int r = 0; r < 8; r++) v[i][r] = at(c + i)[(2 + r0 + r) * 64];
        }
#pragma unroll
        for (int i = 0; i < kMergeAhead; i++) {
            if (c + i < parts) {
                const float f = __builtin_amdgcn_exp2f(v[i][8] - m);
                l += v[i][9] * f;
#pragma unroll
                for (int r = 0; r < 8; r++) o[r] += v[i][r] * f;
            }
        }
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int q = 0; q < 2; q++)
        store_operand4<PAIRS>(p.out, b * p.len + t, h * 64 + r0 * 2 + q * 8 + h32 * 4, p.d_model / kSplitCols, o[4 * q] * inv,
                              o[4 * q + 1] * inv, o[4 * q + 2] * inv, o[4 * q + 3] * inv, p.pair_scale);
}

}  // namespace gh
