// nbx_exact.h - correctly rounded FP64 building blocks of the bit-identical
// paths (all-pairs FP64, exact Barnes-Hut walk), and pair potentials.
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

// 1 / sqrt(x) to about an ulp for normal x (the third-order step alone).
__device__ inline double near_rsqrt(double x) {
    const double y0 = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y0), y0, 1.0);
    return __builtin_fma(y0 * e, __builtin_fma(e, 0.375, 0.5), y0);
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

// ExactGuard for one argument x and divisor p.
__device__ inline bool exact_odd(double x, double p) {
    const unsigned hi = static_cast<unsigned>(__double2hiint(x));
    return (hi - (423u << 20) >= (1200u << 20)) |
           (static_cast<unsigned>(__double2loint(p)) == 0xFFFFFFFFu);
}

// Softened pair potentials m_i m_j / d_ij (numerics.c:83-116) of target i over
// the kPotSources sources from j0, those with i < j < n; MASKED unless all of
// them are. Sources are read through scalar loads, so j0 has to be uniform over
// the wave. The bound is FP64 issue, about 16 operations and one v_rsq_f64 a
// pair: 1 / sqrt comes from that by one third-order step, not from an IEEE
// square root and divide. Where that does not hold (a squared distance below
// the normal range, a sum that is NaN) the IEEE operations form the sum again.
// (4,096 clusters of 64 to 4,096, one wave per 64 targets: 3.4 ms; 9.1 ms with
// the IEEE operations and one source at a time.)
constexpr int kPotSources = 16;

template <bool MASKED>
__device__ inline double pot_unit(const double* __restrict__ px, const double* __restrict__ py,
                                  const double* __restrict__ pz, const double* __restrict__ m,
                                  int n, int j0, int i, double x, double y, double z, double mi,
                                  double eps2) {
    constexpr int K = 4;
    double sum = 0.0;
    unsigned low = 0x7FFFFFFFu;
#pragma unroll
    for (int g = 0; g < kPotSources; g += K) {
        double r2[K], w[K];
#pragma unroll
        for (int e = 0; e < K; ++e) {
            const int j = MASKED ? min(j0 + g + e, n - 1) : j0 + g + e;
            const double dx = px[j] - x;
            const double dy = py[j] - y;
            const double dz = pz[j] - z;
            r2[e] = __builtin_fma(dz, dz, __builtin_fma(dy, dy, __builtin_fma(dx, dx, eps2)));
            w[e] = mi * m[j];
            if (MASKED) {
                const bool on = j0 + g + e > i && j0 + g + e < n;
                r2[e] = on ? r2[e] : 1.0;
                w[e] = on ? w[e] : 0.0;
            }
            low = min(low, static_cast<unsigned>(__double2hiint(r2[e])));
        }
#pragma unroll
        for (int e = 0; e < K; ++e) {
            sum = __builtin_fma(w[e], near_rsqrt(r2[e]), sum);
        }
    }
    if (__builtin_amdgcn_ballot_w64(low < (1u << 20) || sum != sum) != 0) {
        asm volatile("");   // a branch, not a select
        sum = 0.0;
        const int end = min(j0 + kPotSources, n);
        for (int j = j0; j < end; ++j) {
            const double dx = px[j] - x;
            const double dy = py[j] - y;
            const double dz = pz[j] - z;
            const double d = sqrt(dx * dx + dy * dy + dz * dz + eps2);
            sum += j > i ? mi * m[j] / d : 0.0;
        }
    }
    return sum;
}

}  // namespace nbx
