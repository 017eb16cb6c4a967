// Sum of exponentials in 32 bits, for the kernels and for the host program that checks its error.
#pragma once

#ifdef __HIPCC__
#define UCM_EXP_FN __host__ __device__ __forceinline__
#else
#define UCM_EXP_FN inline
#endif

namespace ucm {

// Sum of exp(x) over arguments x from -200 to 0, one of which is 0: terms below 2^-126 may be taken for 0.  exp2(t) is
// the hardware's 2^t.  The exponent t = x log2(e) is rounded to whole steps of up to 2^-17; what that and log2(e)'s own
// rounding took, x - t ln 2 with ln 2 in two words, is at most 8e-6 and goes to first order (3e-11 of a term is left) into
// a sum of its own: added to every term by itself it would be rounded once more.  So a term is as exact as exp2, in eight
// instructions, where one with its exponent carried in two words in front of exp2 takes twelve.
struct ExpSum {
    float s = 0.0f, c = 0.0f;

    template <class Exp2>
    UCM_EXP_FN void add(float x, Exp2 exp2)
    {
        constexpr float kLog2e = 1.44269502f, kLn2 = 0.693147182f, kLn2Low = -1.90465421e-9f;
        const float t = x * kLog2e;
        const float e = exp2(t);
        s += e;
        c = __builtin_fmaf(e, __builtin_fmaf(-t, kLn2Low, __builtin_fmaf(-t, kLn2, x)), c);
    }
    UCM_EXP_FN float sum() const { return s + c; }
};

}  // namespace ucm
