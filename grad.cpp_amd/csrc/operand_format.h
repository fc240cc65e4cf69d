// How matrices whose products are formed of parts are stored: three bf16 parts of an fp32 value
// (kernels_split.h says why they suffice) and two fp16 ones (kernels_pair.h).
#pragma once

#include "kernels_common.h"

namespace gh {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Two floats as three words of two bf16 each (low half: the first float's part).
__device__ __forceinline__ void split_pair(float x, float y, unsigned& p1, unsigned& p2, unsigned& p3) {
    const auto pack = [](float a, float b) {
        return __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{a, b}), v2bf));
    };
    const auto lo = [](unsigned w) { return __uint_as_float(w << 16); };
    const auto hi = [](unsigned w) { return __uint_as_float(w & 0xFFFF0000u); };
    p1 = pack(x, y);
    x -= lo(p1);
    y -= hi(p1);
    p2 = pack(x, y);
    p3 = pack(x - lo(p2), y - hi(p2));
}

constexpr unsigned kSplitTop = 0x7F7F8000u;  // bits of the smallest magnitude that rounds to an infinite bf16

// Storage of a split matrix (rows x K, K a multiple of 16): blocks of 16 rows x 16 columns,
// 1536 contiguous bytes each, row group by row group and inside one along K.  In a block a
// row is 96 bytes: the 16 first parts, the 16 second, the 16 third, each as two 16-byte
// chunks of eight columns, in the other order in rows 8..15.  A block is copied into LDS as
// it is; that exchange of chunks makes the 16-byte operand reads of 16 rows fall on all 64
// banks once.
constexpr int kSplitRows = 16, kSplitCols = 16;
constexpr int kSplitPartBytes = kSplitCols * 2;  // from one part of a row to the next
constexpr int kSplitRowBytes = 3 * kSplitPartBytes;
constexpr int kSplitBlockBytes = kSplitRows * kSplitRowBytes;

// Byte offset of the first part of column k (a multiple of 8: the start of a chunk) of row r.
__device__ __forceinline__ size_t split_offset(int r, int k, int kblocks) {
    return (static_cast<size_t>(r >> 4) * kblocks + (k >> 4)) * kSplitBlockBytes + (r & 15) * kSplitRowBytes
           + ((((k >> 3) & 1) ^ ((r >> 3) & 1)) << 4);
}

// Eight consecutive columns (k a multiple of 8) of one row.
__device__ __forceinline__ void store_split8(char* base, int r, int k, int kblocks, const float (&v)[8]) {
    v4u p1, p2, p3;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned a, b, c;
        split_pair(v[2 * i], v[2 * i + 1], a, b, c);
        p1[i] = a;
        p2[i] = b;
        p3[i] = c;
    }
    char* at = base + split_offset(r, k, kblocks);
    *reinterpret_cast<v4u*>(at) = p1;
    *reinterpret_cast<v4u*>(at + kSplitPartBytes) = p2;
    *reinterpret_cast<v4u*>(at + 2 * kSplitPartBytes) = p3;
}

// Four consecutive columns (k a multiple of 4).
__device__ __forceinline__ void store_split4(char* base, int r, int k, int kblocks, float x, float y, float z, float w) {
    v2u p1, p2, p3;
    unsigned a, b, c;
    split_pair(x, y, a, b, c);
    p1[0] = a, p2[0] = b, p3[0] = c;
    split_pair(z, w, a, b, c);
    p1[1] = a, p2[1] = b, p3[1] = c;
    char* at = base + split_offset(r, k & ~7, kblocks) + (k & 4) * 2;
    *reinterpret_cast<v2u*>(at) = p1;
    *reinterpret_cast<v2u*>(at + kSplitPartBytes) = p2;
    *reinterpret_cast<v2u*>(at + 2 * kSplitPartBytes) = p3;
}

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Storage of a matrix of pairs (rows x K, K a multiple of 16): blocks of 16 rows x 16 columns, 1024
// contiguous bytes each, row group by row group and inside one along K.  A block is the first parts of columns
// 0..7 of its 16 rows (16 bytes each), those of columns 8..15, and the second parts likewise: 16 lanes that read
// an operand's 16 rows read 256 consecutive bytes of LDS.
constexpr int kPairBlockBytes = 1024, kPairPartBytes = 512, kPairChunkBytes = 256;

// Byte offset of the first part of column k (a multiple of 8) of row r.
__device__ __forceinline__ size_t pair_offset(int r, int k, int kblocks) {
    return (static_cast<size_t>(r >> 4) * kblocks + (k >> 4)) * kPairBlockBytes + ((k >> 3) & 1) * kPairChunkBytes + (r & 15) * 16;
}

constexpr float kPairLift = 2048.0f;  // 2^11, of an activation's second part

// Two values as two words of two fp16 each (low half: the first value's part).  The first parts are hidden from the
// compiler once they are made: it would form them a second time, by an instruction that rounds halves the other way, for
// the subtraction.
__device__ __forceinline__ void to_pairs(float x, float y, float lift, unsigned& first, unsigned& second) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    first = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{x, y}), v2h));
    asm("" : "+v"(first));
    const v2h f = __builtin_bit_cast(v2h, first);
    second = __builtin_bit_cast(
        unsigned, __builtin_convertvector((v2f{(x - static_cast<float>(f[0])) * lift, (y - static_cast<float>(f[1])) * lift}), v2h));
}

// Eight consecutive columns (k a multiple of 8) of one row of activations.
__device__ __forceinline__ void store_pair8(char* base, int r, int k, int kblocks, const float (&v)[8], float scale) {
    v4u p1, p2;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned a, b;
        to_pairs(v[2 * i] * scale, v[2 * i + 1] * scale, kPairLift, a, b);
        p1[i] = a;
        p2[i] = b;
    }
    char* at = base + pair_offset(r, k, kblocks);
    *reinterpret_cast<v4u*>(at) = p1;
    *reinterpret_cast<v4u*>(at + kPairPartBytes) = p2;
}

// Four consecutive columns (k a multiple of 4).
__device__ __forceinline__ void store_pair4(char* base, int r, int k, int kblocks, float x, float y, float z, float w, float scale) {
    v2u p1, p2;
    unsigned a, b;
    to_pairs(x * scale, y * scale, kPairLift, a, b);
    p1[0] = a, p2[0] = b;
    to_pairs(z * scale, w * scale, kPairLift, a, b);
    p1[1] = a, p2[1] = b;
    char* at = base + pair_offset(r, k & ~7, kblocks) + (k & 4) * 2;
    *reinterpret_cast<v2u*>(at) = p1;
    *reinterpret_cast<v2u*>(at + kPairPartBytes) = p2;
}

// Four consecutive columns of a row of activations, in the form that the projection behind reads: three parts, or pairs
// scaled by pair_scale.  A kernel is made for either: a condition here would part the values' products from the
// subtractions behind them, and their rounding would go into the parts.
template <bool PAIRS>
__device__ __forceinline__ void store_operand4(char* base, int r, int k, int kblocks, float x, float y, float z, float w,
                                               float pair_scale) {
    if constexpr (PAIRS) store_pair4(base, r, k, kblocks, x, y, z, w, pair_scale);
    else store_split4(base, r, k, kblocks, x, y, z, w);
}

}  // namespace gh
