// Error of ucm::ExpSum's terms against exp in 64 bits, with an exactly rounded 2^t in the place of the hardware's: prints
// "<largest relative error> <mean relative error>" for a million arguments of [lo, 0], or returns 1 where an end of the range is wrong.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>

#include "exp_sum.h"

static float exp2_rounded(float t) { return (float)std::exp2((double)t); }

static double term(float x)
{
    ucm::ExpSum a;
    a.add(x, exp2_rounded);
    return (double)a.s + (double)a.c;
}

int main(int, char** argv)
{
    const float lo = (float)std::atof(argv[1]);
    if (term(0.0f) != 1.0 || term(-200.0f) > 1e-45 || !std::isnan(term(std::numeric_limits<float>::quiet_NaN()))) return 1;
    ucm::ExpSum all;
    for (int i = 0; i < 64; ++i) all.add(0.0f, exp2_rounded);
    if (all.sum() != 64.0f) return 1;
    std::mt19937 gen(7);
    std::uniform_real_distribution<float> of(lo, 0.0f);
    const int n = 1000000;
    double most = 0.0, sum = 0.0;
    for (int i = 0; i < n; ++i) {
        const float x = of(gen);
        const double want = std::exp((double)x), err = (term(x) - want) / want;
        most = std::fmax(most, std::fabs(err));
        sum += err;
    }
    std::printf("%.3e %.3e\n", most, sum / n);
    return 0;
}
