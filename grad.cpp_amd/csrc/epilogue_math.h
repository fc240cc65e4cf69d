// The functions in the epilogues of the products of pairs, of the hardware's 2^x and reciprocal (each within a unit of the
// last place), at the error of tanhf, expf and a division.
//
// Unit: the two instructions; the kernels have the device's, their test on the host ones that are off by as much.
// Error on the device, 2-norm over 2-norm against float64, for normal arguments of spread 0.5 / 1 / 4, those functions -> the two
// instructions alone -> these: GELU 4.1 / 3.8 / 2.2 e-8 -> 4.8 / 4.7 / 2.7 -> 3.0 / 2.7 / 1.6, SiLU 3.8 / 3.9 / 4.2 -> 4.8 / 4.7 /
// 4.6 -> 2.8 / 2.7 / 2.5.  Exponentials of -20 to 0 2.43 -> 3.1 -> 2.45; of that error a sum of thousands keeps what all have in
// common, 2.3 -> 63 -> 2.3 e-9.
#pragma once

#if defined(__HIPCC__)
#define GH_EPILOGUE_FN __device__ __forceinline__
#else
#define GH_EPILOGUE_FN inline
#endif

namespace gh {

template <class Unit>
struct EpilogueMath {
    // x / (1 + e): what 1 + e loses (half a unit of a value near one, for e well below it) and the quotient's own
    // remainder are put back.  e up to 2^126.
    static GH_EPILOGUE_FN float over_one_plus(float x, float e) {
        const float d = 1.0f + e, lost = e - (d - 1.0f), r = Unit::rcp(d), q = x * r;
        return __builtin_fmaf(__builtin_fmaf(-lost, q, __builtin_fmaf(-d, q, x)), r, q);
    }
    // Arguments below 2^40 in size, as pair_bounds has them.
    // 0.5 x (1 + tanh(u)) = x / (1 + exp(-2 u)), u = sqrt(2 / pi) (x + 0.044715 x^3): a negative argument loses nothing to
    // 1 + tanh(u).
    static GH_EPILOGUE_FN float gelu(float x) {
        constexpr float k = -2.0f * 0.79788456f * 1.44269504f;
        return over_one_plus(x, Unit::exp2(__builtin_fminf(x * __builtin_fmaf(x * x, 0.044715f * k, k), 126.0f)));
    }
    // 2^h is exp(t) but for what t log2(e) lost to be h, which is put back behind it.
    static GH_EPILOGUE_FN float silu(float x) {
        const float t = __builtin_fminf(-x, 87.0f), h = t * 1.44269504f, e = Unit::exp2(h);
        return over_one_plus(x, __builtin_fmaf(e, __builtin_fmaf(-h, 0.693147182f, t), e));
    }
    // exp of a logit less the largest: 0 of -inf, NaN of NaN.  2^x of a fraction is off by what the instruction is off by, and
    // whole powers lose nothing.  (Beyond 200 of those the rest counts as fraction, and 2^x of that is 0.)  16384 x 16000 x 768
    // of scored logits 1161 us, as with a product that puts back what x log2(e) loses, whose own rounding made it 2.7; by expf 1212
    // for 1119.
    static GH_EPILOGUE_FN float exp_of(float x) {
        const float n = __builtin_fmaxf(__builtin_rintf(x * 1.44269502f), -200.0f);
        const float part = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, 1.44269502f, -n));  // log2(e) in two parts
        return __builtin_ldexpf(Unit::exp2(part), static_cast<int>(n));
    }
};

}  // namespace gh
