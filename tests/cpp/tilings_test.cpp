// The forms and tilings that tilings.h gives: a line per line of the input.
//   layers D FFN1_OUTPUTS ROWS | logits D VOCAB ROWS          parts or pairs
//   few ROWS OUTPUTS 0|1          fp32 products of few rows, without and with six tiles
//   parts ROWS OUTPUTS K | pairs ROWS OUTPUTS K rows|gelu|swiglu|logits          the tiling
#include "../../grad.cpp_amd/csrc/tilings.h"

#include <cstdio>
#include <cstring>

int main() {
    const char* const split[] = {"32 K4", "64 K4", "64", "128x64", "128"};
    const char* const pair[] = {"128", "128x64", "64", "64 K2", "64x96 K2", "64x96 K4", "32 K4", "quarters"};
    const char* const few[] = {"1x1", "1x2", "2x1", "2x2", "3x2", "2x3"};
    const char* const outs[] = {"rows", "gelu", "swiglu", "logits"};
    char what[16], out[16];
    int a, b, c;
    while (std::scanf("%15s %d %d %d", what, &a, &b, &c) == 4) {
        const bool narrow = a < gh::kPairMinCols;
        if (!std::strcmp(what, "layers")) std::puts(narrow || gh::parts_are_closer(a, b, c) ? "parts" : "pairs");
        else if (!std::strcmp(what, "logits")) std::puts(narrow || gh::logits_parts_are_closer(a, b, c) ? "parts" : "pairs");
        else if (!std::strcmp(what, "few")) std::puts(few[gh::rows_tiles(a, b, c != 0)]);
        else if (!std::strcmp(what, "parts")) std::puts(split[gh::split_tiling(a, b, c)]);
        else if (std::scanf("%15s", out) == 1) {
            int o = 0;
            while (o < 3 && std::strcmp(outs[o], out)) o++;
            std::puts(pair[gh::pair_tiling(a, b, c, static_cast<gh::PairOut>(o))]);
        }
    }
}
