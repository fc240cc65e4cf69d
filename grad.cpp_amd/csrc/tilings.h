// Which form and which tiling a product of many rows takes: rules of sizes, for the host alone.
#pragma once

#include <algorithm>
#include <cmath>

namespace gh {

constexpr int kPairMinCols = 512;  // narrower models have no pairs (kernels_pair.h)

// Products of so many rows and outputs of which split_gemm shares K among four sets of wavefronts (one round of 64 x 64 tiles).
inline bool split_in_four_sets(long rows, long outputs) { return (rows + 63) / 64 * ((outputs + 63) / 64) <= 256; }

// Three parts whose products of few rows are shared among four sets have the smaller errors up to 1024 columns (K = 512
// 0.77e-7 against 1.09, 768 0.88 / 1.12, 1024 0.98 / 1.14; in one set 1.28, 1.59, 1.86), those of longer K never (2048 1.34 /
// 1.20).  Over a layer the wider of its products decide: error of the second layer's values, pairs over three parts, below
// the line and above: GPT-2 512 wide 1.10 (512 rows), 0.98 (513), 768 1.03 (320), 0.88 (321), Llama 768 1.05 (256), 0.98 (300);
// from 1024 on pairs are closer with any rows (160: 0.95).  Below 640 columns q, k, v count too (Llama 512 wide: 1.03 at 640
// rows, 0.97 at 641).
inline bool parts_are_closer(int d_model, int ffn1_outputs, long rows) {
    return d_model < 1024 && (split_in_four_sets(rows, ffn1_outputs) || (d_model < 640 && split_in_four_sets(rows, 3 * d_model)));
}

inline bool logits_parts_are_closer(int d_model, int vocab, long rows) { return d_model <= 1024 && split_in_four_sets(rows, vocab); }

// Three parts: which tiling.  Measured over 14 row counts from 160 to 8192 against five matrices (768
// columns: 768, 2304, 4096 outputs; 2048 columns: 768, 512 outputs), the rule takes the fastest
// tiling or one within 6 % of it:
// - With two 32 x 32 tiles per compute unit at most they win, K shared by four sets of
//   wavefronts, and after them 64 x 64 tiles with K shared the same way: such a launch is a chain
//   of K steps of about 250 ns each (load, LDS, registers, product), so the shorter chain is what
//   counts (1001 x 768 x 2048: 25 us against 35 with K in one set; 160 x 768 x 2048: 11 against 21).
// - With more tiles than compute units the chains hide behind each other.  Tiles are dealt to 256
//   compute units in whole rounds, and a round of 128 x 128 tiles costs 2.8 times one of 64 x 64
//   (four times the products, half the operand bytes per product): the cheaper one
//   (6000 x 768 x 2048: 120 us against 126; 8192 x 4096 x 768: 247, i.e. 208 TFLOP/s of fp32 products
//   or 1.25 PFLOP/s of bf16, against 303).
// - Two rounds of 64 x 64 tiles that are one round of 128 x 64 ones are taken as those, a
//   tile's four stages in flight: a wavefront reads three fragments from LDS for two products
//   instead of four, and no compute unit is left with two tiles where its neighbour has one.  Same
//   sums in the same order.  280 to 510 tiles of 64 x 64, 40 launches (2231 x 768 x 768: 22.2 to
//   20.6 us; 1999 x 768 x 2048: 43.4 to 41.3; 2231 x 768 x 3072: 66.2 to 60.8; 695 x 2304 x 768:
//   21.2 to 20.5): 2 to 8 % faster from 768 columns on, between 11 % slower and 4 % faster at 512, where
//   filling the longer ring is a larger part.  With more tiles than one each they lose (2807 x 768 x 2048:
//   67.8 against 61.3), as do 128 x 64 tiles of eight wavefronts.
enum SplitTiling { SPLIT_32_K4, SPLIT_64_K4, SPLIT_64, SPLIT_128x64, SPLIT_128 };

inline SplitTiling split_tiling(int M, int N, int K) {
    const auto tiles = [&](int t) { return static_cast<long>((M + t - 1) / t) * ((N + t - 1) / t); };
    const auto rounds = [&](int t) { return (tiles(t) + 255) / 256; };
    if (rounds(32) <= 2) return SPLIT_32_K4;
    if (split_in_four_sets(M, N)) return SPLIT_64_K4;
    const long tall = static_cast<long>((M + 127) / 128) * ((N + 63) / 64);
    if (rounds(64) == 2 && tall <= 256 && K >= 768) return SPLIT_128x64;
    return rounds(128) * 28 < rounds(64) * 10 ? SPLIT_128 : SPLIT_64;
}

// Pairs: the tilings, and what a launch takes with each: with n tiles on the fullest of 256 compute units and K in thousands
//   start + max(chain K, n step K) + n out
// us, fitted to 230 launches (160 to 16384 rows against the ten matrices of models 512 and 768 columns wide: W_o, QKV,
// both FFN1 and FFN2), medians off by 2 to 5 %.  A lone workgroup is a chain of K steps (64 x 64 tiles with K shared by
// two sets of wavefronts, and 32 x 32 ones by four, are the shorter chains); beside others its chain hides, and what
// counts is what the unit moves through LDS and multiplies; `out` is the epilogue, of a residual (queries, keys, values
// and logits counted like it), a GELU or a SwiGLU.  Taking the least by this rule, those launches take 0.8 % longer
// than with the best of the seven tilings each (at most 18 %), by the three-part form's rule 5.1 (at most 44 %): 1999 x
// 768 x 768 14.0 -> 11.4 us, 1999 x 768 x 2048 31.9 -> 24.2, 1999 x 2304 x 768 31.8 -> 31.1, 1999 x 3072 x 768 37.5 ->
// 34.8.  (Four tilings more, among them 96 x 192, 192 x 64 and 128 x 96, were the best by less than 1 % together.)
struct PairTilingTime {
    int m, n, sets;  // rows, outputs, sets of wavefronts that share K
    float start, chain, step, out[3];
};
enum PairTiling { PAIR_128, PAIR_128x64, PAIR_64, PAIR_64_K2, PAIR_64x96_K2, PAIR_64x96_K4, PAIR_32_K4, PAIR_MIXED };
enum PairOut { PAIR_ROWS, PAIR_GELU, PAIR_SWIGLU, PAIR_LOGITS };
constexpr PairTilingTime kPairTilings[PAIR_MIXED] = {
    {128, 128, 1, 1.64f, 21.42f, 18.17f, {4.43f, 4.01f, 3.31f}}, {128, 64, 1, 2.15f, 13.10f, 10.78f, {1.94f, 1.80f, 1.20f}},
    {64, 64, 1, 1.90f, 9.58f, 6.45f, {1.00f, 0.80f, 0.58f}},     {64, 64, 2, 1.61f, 6.59f, 6.31f, {1.18f, 1.18f, 1.01f}},
    {64, 96, 2, 2.37f, 10.21f, 8.57f, {2.15f, 2.14f, 1.44f}},    {64, 96, 4, 0.50f, 2.40f, 8.44f, {3.72f, 4.87f, 3.85f}},
    {32, 32, 4, 2.14f, 2.68f, 2.53f, {0.46f, 0.81f, 0.62f}},
};

// PAIR_MIXED: 128 x 128 tiles in whole rounds of 256 and the rest, at most 64 of them, as 64 x 64 quarters in the same
// launch, at most one for each compute unit, beside its last whole tile (both fit it).  2000 x 2304 outputs are 288
// tiles: 32 compute units had two and the others waited.  Of 230 launches (160 to 16384 rows) the rule gives it 18, all
// of them faster than what they took before, by 7 to 22 % (1999 x 2304 x 768 33.0 -> 28.6 us, in a prompt 37.5 -> 32.4,
// 6000 x 768 x 2048 67.8 -> 61.3, 1280 x 4096 x 768 32.2 -> 27.1, 7000 x 3072 x 768 111.0 -> 101.3); with more than one
// quarter for a compute unit it is the slower one in 32 of 45 (2600 x 3072 x 768 42.4 -> 48.6, 1800 x 4096 x 768 38.2
// -> 44.0).  Not for scored logits, whose sums of exponentials are kept for 64 columns at a time.
constexpr int kPairMixedRest = 64;

inline PairTiling pair_tiling(int M, int N, int K, PairOut what) {
    const int out = what == PAIR_LOGITS ? PAIR_ROWS : what;
    PairTiling best = PAIR_128;
    float least = INFINITY;
    for (int i = 0; i < PAIR_MIXED; i++) {
        const PairTilingTime& t = kPairTilings[i];
        if (K % (64 * t.sets) != 0) continue;  // (whole parts per set)
        const float tiles = static_cast<float>((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n), n = std::ceil(tiles / 256.0f);
        const float us = t.start + std::max(t.chain, n * t.step) * K * 1e-3f + n * t.out[out];
        if (us < least) {
            least = us;
            best = static_cast<PairTiling>(i);
        }
    }
    const int tiles = (M + 127) / 128 * ((N + 127) / 128), rounds = tiles / 256, rest = tiles % 256;
    if (what != PAIR_LOGITS && rounds > 0 && rest > 0 && rest <= kPairMixedRest) {
        const PairTilingTime &a = kPairTilings[PAIR_128], &b = kPairTilings[PAIR_64];
        const float us = a.start + std::max(a.chain, rounds * a.step + b.step) * K * 1e-3f + rounds * a.out[out] + b.out[out];
        if (us < least) best = PAIR_MIXED;
    }
    return best;
}

// fp32 products of 65 to 511 rows in tiles of 16 x 16 (gemm16_kernel on eight wavefronts): how many of them, rows x outputs, a
// workgroup takes.  A launch costs a start and then, for every workgroup that a compute unit is dealt, a time that grows
// more slowly than the tiles in it, since more tiles share the rows they read (what is being paid for is operand traffic
// from the L2s and operand permutes, 2 x 2 tiles having half of both per product): per workgroup and 768 columns 1 x 1
// tiles 1.7 us, two 2.4 or 2.5, 2 x 2 4.0, 3 x 2 5.9, 2 x 3 6.2.  Runs of outputs are dealt to the eight XCDs in turn,
// each with all its rows (the weights stay in that L2), so what counts is the XCD with the most of them over its 32
// compute units: 511 x 576 in 3 x 2 tiles are 198 workgroups and yet two rounds on an XCD that has 3 of the 18 runs
// (K = 2304 32.9 us; 2 x 3 20.4).  Over 784 launches (16 row counts against W_o, FFN1 and FFN2 of 13 widths from 512 to 1536) the
// rule takes 1.3 % longer than the best of the six each; with the workgroups counted over the whole chip 3.8 %, 62 % at most
// (397 x 896 x 3584 48.5 us against 29.9), and 4.7 % without 3 x 2 and 2 x 3, which are there for row counts where
// four tiles leave a last workgroup to few compute units (511 x 768 x 768 11.2 -> 9.5, 397 x 768 x 2048 19.5 -> 18.0).
// Queries, keys and values stay with four: six tiles are a second round of their epilogue, whose reads (position,
// page, rotation) nothing hides (244 x 2304 x 768 in a prompt 20.2 us -> 23.4).
// (profiles/many_row_tilings.md.  Both operands through an LDS ring, 32 x 32 to 64 x 64 outputs per workgroup: 35-36 us at
// 397 x 4096 x 768, slower than this at every narrower shape.)
enum RowsTiles { ROWS_1x1, ROWS_1x2, ROWS_2x1, ROWS_2x2, ROWS_3x2, ROWS_2x3 };
struct RowsTilesTime {
    int rows, outputs, each;  // 16-row tiles, 16-output tiles, a workgroup's time
};

inline RowsTiles rows_tiles(int M, int N, bool six) {
    const bool wide = N > 1024;
    const RowsTilesTime tiles[] = {{1, 1, 17}, {1, 2, wide ? 24 : 25}, {2, 1, wide ? 25 : 24}, {2, 2, 40}, {3, 2, 59}, {2, 3, 62}};
    const auto cost = [&](RowsTiles t) {
        const long row_groups = (M + 16 * tiles[t].rows - 1) / (16 * tiles[t].rows);
        const long runs = (N + 16 * tiles[t].outputs - 1) / (16 * tiles[t].outputs);
        return ((runs + 7) / 8 * row_groups + 31) / 32 * tiles[t].each;
    };
    RowsTiles best = ROWS_2x2;  // (of equals the more tiles, but four before six)
    for (const RowsTiles t : {ROWS_1x2, ROWS_2x1, ROWS_1x1})
        if (cost(t) < cost(best)) best = t;
    if (six) {
        for (const RowsTiles t : {ROWS_3x2, ROWS_2x3})
            if (cost(t) < cost(best)) best = t;
    }
    return best;
}

}  // namespace gh
