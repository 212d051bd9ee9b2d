// nbx_exact.h - correctly rounded FP64 building blocks of the bit-identical
// paths (all-pairs FP64, exact Barnes-Hut walk).
//
// The reference's pair term needs RN(1 / RN(sqrt(x))) (gravity.c:52-53), its
// walk RN(1 / RN(x RN(sqrt(x)))) (barnes_hut.c:595-598), RN = round to nearest
// even. The compiler's IEEE sqrt and divide each scale their operand for the
// whole exponent range and take a transcendental of their own. Here one
// v_rsq_f64 (relative error 2^-24.2 measured over 4M values of [1, 4)) feeds
// both, without scaling, where the argument is well inside the exponent range:
//  - y = 1 / sqrt(x) by one step of third order, y0 (1 + e / 2 + 3 e^2 / 8)
//    with e = 1 - x y0^2: what is left is the step's own rounding;
//  - square root: g = x y, then g + (x - g^2) y / 2, whose residual an FMA
//    gives exactly, rounds to RN(sqrt(x));
//  - reciprocal: two Newton steps y += y (1 - s y). The last residual is
//    exact, and RN(y + y e) is RN(1 / s) for every s whose significand is not
//    all ones (P. Markstein, Computation of elementary functions on the IBM
//    RISC System/6000 processor, IBM J. Res. Dev. 34, 1990).
// ExactGuard collects the arguments outside 2^-600 .. 2^600 (zero, infinities
// and NaN among them) and the divisors whose low significand word is all
// ones; where odd() says so, the caller takes the IEEE operations instead.
#pragma once

#include <hip/hip_runtime.h>

namespace nbx {

struct ExactGuard {
    unsigned hi_max = 0u, hi_min = 0x7FFFFFFFu, lo_max = 0u;

    __device__ void argument(double x) {
        const unsigned hi = static_cast<unsigned>(__double2hiint(x));
        hi_max = max(hi_max, hi);
        hi_min = min(hi_min, hi);
    }
    __device__ void divisor(double s) {
        lo_max = max(lo_max, static_cast<unsigned>(__double2loint(s)));
    }
    // exponent fields 423 .. 1622 (a set sign bit makes hi_max larger)
    __device__ bool odd() const {
        return (hi_max >= (1623u << 20)) | (hi_min < (423u << 20)) | (lo_max == 0xFFFFFFFFu);
    }
};

// s = RN(sqrt(x)); y ~ 1 / sqrt(x) to about an ulp.
__device__ inline double exact_sqrt(double x, double& y) {
    const double y0 = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y0), y0, 1.0);
    y = __builtin_fma(y0 * e, __builtin_fma(e, 0.375, 0.5), y0);
    const double g = x * y;
    return __builtin_fma(__builtin_fma(-g, g, x), 0.5 * y, g);
}

// RN(1 / s) from an approximation y of 1 / s.
__device__ inline double exact_recip(double s, double y) {
    y = __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
}

// RN(1 / RN(sqrt(x))) unless guard.odd().
__device__ inline double exact_inv_sqrt(double x, ExactGuard& guard) {
    double y;
    const double s = exact_sqrt(x, y);
    guard.argument(x);
    guard.divisor(s);
    return exact_recip(s, y);
}

}  // namespace nbx
