// Errors of the epilogues' functions (epilogue_math.h) over those of tanhf, expf and a division, with a 2^x and a reciprocal that
// are off by up to a unit of the last place, as the hardware's are.  Prints name, spread, error over error.
#include "../../grad.cpp_amd/csrc/epilogue_math.h"

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <functional>
#include <random>

// the float next below or next above, as its bits have it
static float faithful(double v) {
    float f = static_cast<float>(v);
    if (f == static_cast<double>(v) || !std::isfinite(f)) return f;
    uint32_t bits;
    std::memcpy(&bits, &f, 4);
    const float other = std::nextafterf(f, f < v ? INFINITY : -INFINITY);
    return (bits * 2654435761u >> 29) < 3 ? other : f;
}

struct HostUnit {
    static float exp2(float x) { return faithful(std::exp2(static_cast<double>(x))); }
    static float rcp(float x) { return faithful(1.0 / static_cast<double>(x)); }
};
using M = gh::EpilogueMath<HostUnit>;

static float gelu_tanh(float x) { return 0.5f * x * (1.0f + std::tanh(0.79788456f * (x + 0.044715f * x * x * x))); }
static float silu_div(float x) { return x / (1.0f + std::exp(-x)); }

int main() {
    const auto over = [](const char* name, double spread, std::function<float(float)> f, std::function<float(float)> g,
                         std::function<double(double)> exact) {
        std::mt19937 rng(7);
        std::normal_distribution<float> normal;
        double a = 0.0, b = 0.0;
        for (int i = 0; i < 400000; i++) {
            const float x = normal(rng) * static_cast<float>(spread);
            const double e = exact(x);
            a += (f(x) - e) * (f(x) - e);
            b += (g(x) - e) * (g(x) - e);
        }
        std::printf("%s %g %.4f\n", name, spread, std::sqrt(a / b));
    };
    for (const double spread : {0.1, 0.5, 1.0, 2.0, 4.0, 16.0}) {
        over("gelu", spread, M::gelu, gelu_tanh,
             [](double x) { return x / (1.0 + std::exp(-2.0 * 0.79788456 * (x + 0.044715 * x * x * x))); });
        over("silu", spread, M::silu, silu_div, [](double x) { return x / (1.0 + std::exp(-x)); });
    }
    // exponentials: their error over that of an exponential as far off as 2^x, and their common relative error, in 1e-9
    std::mt19937 rng(9);
    double own = 0.0, unit = 0.0, common = 0.0;
    for (int i = 0; i < 400000; i++) {
        const float x = -20.0f * (rng() >> 8) / 16777216.0f;
        const double e = std::exp(static_cast<double>(x)), off = M::exp_of(x) / e - 1.0, least = faithful(e) / e - 1.0;
        own += off * off;
        unit += least * least;
        common += off / 400000 * 1e9;
    }
    std::printf("exp %.4f\ncommon exp %.3f\n", std::sqrt(own / unit), common);
    // the ends: what the functions themselves give there
    for (const float x : {-INFINITY, -1e30f, -200.0f, 0.0f, static_cast<float>(std::nan(""))}) std::printf("ends exp %g\n", M::exp_of(x));
    for (const float x : {-1e12f, -200.0f, 0.0f, 200.0f, 1e12f, static_cast<float>(std::nan(""))})
        std::printf("ends gelu %g silu %g\n", M::gelu(x), M::silu(x));
}
