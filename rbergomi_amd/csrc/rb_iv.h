// rb_iv.h -- implied vol of one option by a whole workgroup of 256 threads.
//
// implied_vol_f64 solves an option in one thread: a bracket, bisection and Newton steps of two
// erfc each, about 25 microseconds of dependent instructions with the rest of the chip idle.  Here the
// workgroup evaluates 256 vols at a time, so that two rounds narrow the bracket to 3e-4 of its
// place, and two or three third-order steps reach the root.
#pragma once
#include <hip/hip_runtime.h>

#include "rb_device.h"

namespace rb {

struct IvShared {
    double s1[256], s2[256];
    int first[4];
};

// the sums of a and b over the workgroup (fixed tree), in every thread
__device__ __forceinline__ void block_sum_pair(double& a, double& b, IvShared& sh) {
    const int t = threadIdx.x;
    sh.s1[t] = a;
    sh.s2[t] = b;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (t < off) {
            sh.s1[t] += sh.s1[t + off];
            sh.s2[t] += sh.s2[t + off];
        }
        __syncthreads();
    }
    a = sh.s1[0];
    b = sh.s2[0];
    __syncthreads();
}

// BS price of the out-of-the-money side at total vol st (bs_price_f64)
__device__ __forceinline__ double bs_total_vol(double lnK, double K, double st, bool call) {
    const double d1 = (-lnK + 0.5 * st * st) / st, d2 = d1 - st;
    return call ? phi_f64(d1) - K * phi_f64(d2) : -phi_f64(-d1) + K * phi_f64(-d2);
}

// the first of the workgroup's 256 predicates that holds (256: none)
__device__ __forceinline__ int block_first(bool up, IvShared& sh) {
    const unsigned long long b = __ballot(up);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh.first[w] = b ? 64 * w + __ffsll(b) - 1 : 256;
    __syncthreads();
    const int f = min(min(sh.first[0], sh.first[1]), min(sh.first[2], sh.first[3]));
    __syncthreads();
    return f;
}

// The value of implied_vol_f64 (to its convergence, |dsigma| <= 1e-14 sigma), every thread of the
// workgroup with the same arguments.  Total vols from 2^-24 to 2^6 are searched on a geometric grid;
// a root outside, or one the steps leave the bracket for, is left to implied_vol_f64 itself, and so
// are vols near its upper limit of 1e6.
__device__ inline double implied_vol_block(double price, double K, double lnK, double tau, IvShared& sh) {
    bool call = true;
    double target = price;
    if (1.0 > K) {
        call = false;
        target = price - 1.0 + K;
    }
    const double upper = call ? 1.0 : K;
    if (!(target > 0.0) || !(target < upper) || !(tau > 0.0)) return __builtin_nan("");
    const int t = threadIdx.x;
    constexpr double STEP = 30.0 / 255.0;
    const double g = exp2(-24.0 + STEP * t);
    const int f = block_first(bs_total_vol(lnK, K, g, call) >= target, sh);
    if (f == 0 || f == 256) return implied_vol_f64(price, K, tau);
    double lo = exp2(-24.0 + STEP * (f - 1)), hi = exp2(-24.0 + STEP * f);
    const double w = (hi - lo) / 257.0;
    const int f2 = block_first(bs_total_vol(lnK, K, lo + w * (t + 1), call) >= target, sh);
    hi = f2 == 256 ? hi : lo + w * (f2 + 1);
    lo = lo + w * f2;
    double s = 0.5 * (lo + hi);
    const double l0 = lo - 2.0 * w, h0 = hi + 2.0 * w;
    for (int it = 0; it < 6; ++it) {
        // Halley's step of f(s) = price(s) - target: f'' / f' = d1 d2 / s
        const double d1 = (-lnK + 0.5 * s * s) / s, d2 = d1 - s;
        const double y = (call ? phi_f64(d1) - K * phi_f64(d2) : -phi_f64(-d1) + K * phi_f64(-d2)) - target;
        const double vega = exp(-0.5 * d1 * d1) * 0.3989422804014327;
        const double nt = y / vega;
        const double ds = nt / (1.0 - 0.5 * nt * (d1 * d2 / s));
        s -= ds;
        if (!(s > l0 && s < h0)) return implied_vol_f64(price, K, tau);
        if (fabs(ds) <= 1e-14 * s) break;
    }
    const double sigma = s / sqrt(tau);
    return sigma < 2e5 ? sigma : implied_vol_f64(price, K, tau);
}

}  // namespace rb
