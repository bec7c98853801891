// rb_math64.h -- FP64 elementary functions of the FP64 pricing kernels (gfx950).
//
// What bounds those kernels is the vector issue of FP64 instructions (1.9 ns per wave64
// instruction and SIMD, against 1.0 for FP32), so the functions here carry only what their
// arguments need: no special cases that cannot occur, the scale factors of the model folded into
// the tables, and 32- and 64-entry tables (in LDS) in place of longer polynomials.  The
// polynomials are Chebyshev interpolants or Lawson-weighted least-squares fits made in 50 digits;
// errors (checked against long double on the host, tests/test_math64_cpu.py, and the device, tests/test_gpu_math64.py) stay at one to two
// units in the last place.  Host and device compile the same code, except that the host uses the
// library's square root and division where the device refines v_rsq_f64 and v_rcp_f64.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "rb_device.h"

namespace rb {

// 2^(j/32)
static constexpr double EXP2_TAB[32] = {
    0x1.0000000000000p+0, 0x1.059b0d3158574p+0, 0x1.0b5586cf9890fp+0, 0x1.11301d0125b51p+0,
    0x1.172b83c7d517bp+0, 0x1.1d4873168b9aap+0, 0x1.2387a6e756238p+0, 0x1.29e9df51fdee1p+0,
    0x1.306fe0a31b715p+0, 0x1.371a7373aa9cbp+0, 0x1.3dea64c123422p+0, 0x1.44e086061892dp+0,
    0x1.4bfdad5362a27p+0, 0x1.5342b569d4f82p+0, 0x1.5ab07dd485429p+0, 0x1.6247eb03a5585p+0,
    0x1.6a09e667f3bcdp+0, 0x1.71f75e8ec5f74p+0, 0x1.7a11473eb0187p+0, 0x1.82589994cce13p+0,
    0x1.8ace5422aa0dbp+0, 0x1.93737b0cdc5e5p+0, 0x1.9c49182a3f090p+0, 0x1.a5503b23e255dp+0,
    0x1.ae89f995ad3adp+0, 0x1.b7f76f2fb5e47p+0, 0x1.c199bdd85529cp+0, 0x1.cb720dcef9069p+0,
    0x1.d5818dcfba487p+0, 0x1.dfc97337b9b5fp+0, 0x1.ea4afa2a490dap+0, 0x1.f50765b6e4540p+0};

// (c_j, 2 ln c_j): c_j is 1 / m to 14 bits at the middle of m in [(64 + j) / 128, (65 + j) / 128),
// and exactly 1 in the last interval, so that logarithms near ln 1 keep their relative accuracy
static constexpr double LOG_TAB[128] = {
    0x1.fc08000000000p+0, 0x1.5ee83aa241520p+0,
    0x1.f448000000000p+0, 0x1.5709526b0286dp+0,
    0x1.ecc0000000000p+0, 0x1.4f45283594e19p+0,
    0x1.e574000000000p+0, 0x1.47a1aa7e829d3p+0,
    0x1.de5c000000000p+0, 0x1.40183a11c698ep+0,
    0x1.d77c000000000p+0, 0x1.38aec9717bde8p+0,
    0x1.d0cc000000000p+0, 0x1.315e5c431f58cp+0,
    0x1.ca4c000000000p+0, 0x1.2a286ed0b7808p+0,
    0x1.c3f8000000000p+0, 0x1.2309fd8ba3896p+0,
    0x1.bdd4000000000p+0, 0x1.1c08fc9a5bf0bp+0,
    0x1.b7d8000000000p+0, 0x1.151daf6ea5216p+0,
    0x1.b204000000000p+0, 0x1.0e495060fbbe2p+0,
    0x1.ac58000000000p+0, 0x1.078d2052e216ap+0,
    0x1.a6d0000000000p+0, 0x1.00e58e5b1f7abp+0,
    0x1.a16c000000000p+0, 0x1.f4a76edf05723p-1,
    0x1.9c2c000000000p+0, 0x1.e7b17c3cf3b6dp-1,
    0x1.9710000000000p+0, 0x1.daeb94828762fp-1,
    0x1.9210000000000p+0, 0x1.ce43b18052743p-1,
    0x1.8d30000000000p+0, 0x1.c1c5c693f839ep-1,
    0x1.8870000000000p+0, 0x1.b573e04220923p-1,
    0x1.83c8000000000p+0, 0x1.a93af3c6cd1d0p-1,
    0x1.7f40000000000p+0, 0x1.9d31bea13ed3bp-1,
    0x1.7ad4000000000p+0, 0x1.914f96328b4b5p-1,
    0x1.767c000000000p+0, 0x1.85806773d09d3p-1,
    0x1.7244000000000p+0, 0x1.79e67685bf954p-1,
    0x1.6e20000000000p+0, 0x1.6e626e6aa9973p-1,
    0x1.6a14000000000p+0, 0x1.6300c0b3a0a49p-1,
    0x1.6620000000000p+0, 0x1.57c2f53b05209p-1,
    0x1.6240000000000p+0, 0x1.4c9f09e152c3cp-1,
    0x1.5e74000000000p+0, 0x1.4196323a2a69cp-1,
    0x1.5ac0000000000p+0, 0x1.36b5776bc1117p-1,
    0x1.5720000000000p+0, 0x1.2bf287cc41362p-1,
    0x1.5390000000000p+0, 0x1.214296d0898d2p-1,
    0x1.5014000000000p+0, 0x1.16b2bcb9a396ap-1,
    0x1.4cac000000000p+0, 0x1.0c444675d40e4p-1,
    0x1.4954000000000p+0, 0x1.01ec15623f492p-1,
    0x1.460c000000000p+0, 0x1.ef563e4c79bdep-2,
    0x1.42d8000000000p+0, 0x1.db1e1b06b799ap-2,
    0x1.3fb0000000000p+0, 0x1.c6ff3c6efcf71p-2,
    0x1.3c98000000000p+0, 0x1.b314c570f3e05p-2,
    0x1.3990000000000p+0, 0x1.9f60c068455e5p-2,
    0x1.3698000000000p+0, 0x1.8be53eb17ee7cp-2,
    0x1.33b0000000000p+0, 0x1.78a4584c00cf2p-2,
    0x1.30d0000000000p+0, 0x1.656a6be1dd2d9p-2,
    0x1.2e04000000000p+0, 0x1.52897e425f200p-2,
    0x1.2b40000000000p+0, 0x1.3fb25a59528cbp-2,
    0x1.288c000000000p+0, 0x1.2d1cf0c573d55p-2,
    0x1.25e4000000000p+0, 0x1.1aaf97d7e33dcp-2,
    0x1.2344000000000p+0, 0x1.084fab53cb5b6p-2,
    0x1.20b4000000000p+0, 0x1.ec6d582f6891bp-3,
    0x1.1e30000000000p+0, 0x1.c8948014bcb6ap-3,
    0x1.1bb4000000000p+0, 0x1.a4de24086f427p-3,
    0x1.1944000000000p+0, 0x1.818622ea35b7cp-3,
    0x1.16e0000000000p+0, 0x1.5e8fa4d8591c7p-3,
    0x1.1484000000000p+0, 0x1.3bc29a634a475p-3,
    0x1.1234000000000p+0, 0x1.195c7d0380c61p-3,
    0x1.0ff0000000000p+0, 0x1.eec11bf25b908p-4,
    0x1.0db4000000000p+0, 0x1.ab2aacd860545p-4,
    0x1.0b80000000000p+0, 0x1.67f94f094bd98p-4,
    0x1.0954000000000p+0, 0x1.2530b2f8c883fp-4,
    0x1.0734000000000p+0, 0x1.c6a22e719902fp-5,
    0x1.0518000000000p+0, 0x1.42cc921478887p-5,
    0x1.0308000000000p+0, 0x1.81b889ebf9f2dp-6,
    0x1.0000000000000p+0, 0x0.0p+0};

constexpr int EXP2_N = 32, LOG_N = 64;
constexpr double EXP2_SCALE = 46.166241308446828384;  // 32 log2(e): exp(x) = 2^(x EXP2_SCALE / 32)

// A whole number as an integer, the nearest end of the range beyond it and 0 for NaN.  C++ leaves int(n)
// undefined there, and every step past a path's last one comes with an exponent of -1e10 and less; the instruction
// is the one int(n) would be, by name (-fno-strict-float-cast-overflow puts six more around it).
__host__ __device__ __forceinline__ int whole_i32(double n) {
#if defined(__HIP_DEVICE_COMPILE__)
    int k;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(n));
    return k;
#else
    return n >= 2147483647.0 ? 2147483647 : n > -2147483648.0 ? int(n) : n <= -2147483648.0 ? -2147483647 - 1 : 0;
#endif
}

// 2^(y / 32): y = n + f with n whole and |f| <= 1/2, 2^(n/32) from the table and an exponent
// shift, 2^(f/32) = 1 + f q(f) with q of degree 4 (relative error 9e-17).  y beyond the exponent
// range gives 0 or infinity (the conversion to an integer saturates); NaN and infinities give NaN.
__host__ __device__ __forceinline__ double exp2_32(const double* T, double y) {
    const double n = rint(y), f = y - n;
    const int k = whole_i32(n);
    double q = fma(0x1.5d8789d24d3fep-35, f, 0x1.3b2b276cebac8p-27);
    q = fma(q, f, 0x1.c6b08d70b74e4p-20);
    q = fma(q, f, 0x1.ebfbdff8098e8p-13);
    q = fma(q, f, 0x1.62e42fefa39edp-6);
    const double t = T[k & (EXP2_N - 1)];
    return ldexp(fma(t * f, q, t), k >> 5);
}

// -2 ln u of u = (x + 1/2) 2^-32: X = 2 x + 1 = m 2^e exactly (m in [1/2, 1)), r = m c_j - 1 exactly
// (33 by 15 bits, |r| <= 1/128), ln u = (e - 33) ln 2 - ln c_j + ln(1 + r),
// ln(1 + r) = r - r^2 (1/2 - ...) with a polynomial of degree 5 (absolute error 4e-18 r)
__host__ __device__ __forceinline__ double neg2_log_u32(const double2* T, uint32_t x) {
    const double X = fma(double(x), 2.0, 1.0);
    uint64_t b;
    __builtin_memcpy(&b, &X, 8);
    const uint32_t hi = uint32_t(b >> 32);
    const int e = int(hi >> 20) - (1022 + 33);
    b = (b & 0xffffffffu) | (uint64_t((hi & 0xfffffu) | 0x3fe00000u) << 32);
    double m;
    __builtin_memcpy(&m, &b, 8);
    const double2 c = T[(hi >> 14) & (LOG_N - 1)];
    const double r = fma(m, c.x, -1.0);
    const double r2 = r * r;
    double p = fma(-0x1.2499c540c351fp-2, r, 0x1.555c556bd5cffp-2);
    p = fma(p, r, -0x1.999999861608bp-2);
    p = fma(p, r, 0x1.fffffff1ffd68p-2);
    p = fma(p, r, -0x1.55555555555cep-1);
    p = fma(p, r, 0x1.000000000001cp+0);
    const double a = fma(double(e), -1.3862943611198906188, c.y);
    return fma(r2, p, fma(-2.0, r, a));
}

// square root of a positive normal number: Goldschmidt steps from v_rsq_f64, the last one on the
// exact residual
__host__ __device__ __forceinline__ double sqrt_pos(double w) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(w);
    double g = w * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    return fma(fma(-g, g, w), h, g);
#else
    return sqrt(w);
#endif
}

// 1 / d of a normal number: two Newton steps from v_rcp_f64
__host__ __device__ __forceinline__ double rcp_pos(double d) {
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(d);
    y = fma(y, fma(-d, y, 1.0), y);
    return fma(y, fma(-d, y, 1.0), y);
#else
    return 1.0 / d;
#endif
}

// Box-Muller on u = (x + 1/2) 2^-32: (r cos 2 pi u1, r sin 2 pi u1), r = sqrt(-2 ln u0).  The
// angle is reduced on the integer: the nearest quarter turn n and the exact remainder
// t = (x1 + 1/2) 2^-30 - n in [-1/2, 1/2] quarter turns; sin and cos of (pi/2) t by polynomials of
// degree 6 in t^2.
__host__ __device__ __forceinline__ void box_muller_f64(const double2* T, uint32_t x0, uint32_t x1, double& z0,
                                                        double& z1) {
    const double r = sqrt_pos(neg2_log_u32(T, x0));
    const uint32_t n = (x1 + 0x20000000u) >> 30;
    const double t = fma(double(int32_t(x1 - (n << 30))), 0x1p-30, 0x1p-31);
    const double s = t * t;
    double ps = fma(0x1.e3f38399551bfp-25, s, -0x1.e30071afc3e59p-19);
    double pc = fma(-0x1.b2f3eb054afcdp-28, s, 0x1.f9ce245cada0bp-22);
    ps = fma(ps, s, 0x1.50782fda12d96p-13);
    pc = fma(pc, s, -0x1.a6d1eef479be1p-16);
    ps = fma(ps, s, -0x1.32d2cce2e5b19p-8);
    pc = fma(pc, s, 0x1.e1f5068688d5bp-11);
    ps = fma(ps, s, 0x1.466bc677587f8p-4);
    pc = fma(pc, s, -0x1.55d3c7e3cb241p-6);
    ps = fma(ps, s, -0x1.4abbce625be41p-1);
    pc = fma(pc, s, 0x1.03c1f081b5ac0p-2);
    ps = fma(ps, s, 0x1.921fb54442d18p+0);
    pc = fma(pc, s, -0x1.3bd3cc9be45dep+0);
    const double sn = (r * t) * ps, cs = fma(r * s, pc, r);
    // quarter turns: n = 0 (c, s), 1 (-s, c), 2 (-c, -s), 3 (s, -c)
    const bool odd = n & 1;
    const double a = odd ? sn : cs, b = odd ? cs : sn;
    uint64_t ua, ub;
    __builtin_memcpy(&ua, &a, 8);
    __builtin_memcpy(&ub, &b, 8);
    ua ^= uint64_t(((n + 1) << 30) & 0x80000000u) << 32;
    ub ^= uint64_t((n << 30) & 0x80000000u) << 32;
    __builtin_memcpy(&z0, &ua, 8);
    __builtin_memcpy(&z1, &ub, 8);
}

// Four normals of path p, stream s, steps 4q .. 4q + 3
__host__ __device__ __forceinline__ void normals4_f64(const double2* T, PhiloxKey key, uint64_t p, uint32_t s,
                                                      uint32_t q, double z[4]) {
    const uint4 x = philox_block(key, p, s, q);
    box_muller_f64(T, x.x, x.y, z[0], z[1]);
    box_muller_f64(T, x.z, x.w, z[2], z[3]);
}

// Mills ratio (1 - Phi(x)) / phi(x) = g(u) / (x + k), u = (x - k) / (x + k), k = 4.5: g on [-1, 1]
// as a polynomial of degree 22 (relative error 2.2e-16)
static constexpr double MILLS_POLY[23] = {
    0x1.e9c33ae3cff7cp+0, -0x1.9ad9f411c9569p+0, 0x1.1e7cb715a38f2p+0,
    -0x1.44e16e0a81f03p-1, 0x1.1de53b9269ca2p-2, -0x1.5bc3103f2e5bdp-4,
    0x1.5aea6f0e9b15fp-7, 0x1.1f49bf1c3d987p-8, -0x1.2d86455731db5p-9,
    0x1.0c5c5dc113585p-16, 0x1.267df5a9298e2p-12, -0x1.4f0a76116188ep-15,
    -0x1.2b580320a0bfep-15, 0x1.0c7b99a45c04cp-17, 0x1.688cbfd68a0b9p-18,
    -0x1.52fc9b5f832cdp-20, -0x1.ff7d4334e1c89p-21, 0x1.63c34948896b4p-23,
    0x1.7f551c7308199p-23, -0x1.0a7a163bf0958p-26, -0x1.ef90d94bff569p-26,
    0x1.73593d9b065c3p-31, 0x1.77b6c9a1ffe4dp-29};

// The Mills ratios of x, y in [0, 1e4], two independent chains on one reciprocal
template <class P = const double*>
__host__ __device__ __forceinline__ void mills_pair(double x, double y, double& mx, double& my, P c = MILLS_POLY) {
    constexpr double k = 4.5;
    const double dx = x + k, dy = y + k, inv = rcp_pos(dx * dy);
    const double ix = inv * dy, iy = inv * dx;
    const double u = (x - k) * ix, w = (y - k) * iy;
    double a = c[22], b = c[22];
#pragma unroll
    for (int i = 21; i >= 0; --i) {
        a = fma(a, u, c[i]);
        b = fma(b, w, c[i]);
    }
    mx = a * ix;
    my = b * iy;
}

// The fields of a path that its options share: ln S', S', sigma = sqrt((1 - rho^2) Iv), 1 / sigma
struct PathRt64 {
    double lnS, S, sig, isig;
};
__host__ __device__ __forceinline__ PathRt64 path_rt64(double Iv, double Is, double rho) {
    PathRt64 q;
    q.sig = sqrt((1.0 - rho * rho) * Iv);
    q.isig = 1.0 / q.sig;
    q.lnS = -0.5 * rho * rho * Iv + rho * Is;
    q.S = exp(q.lnS);
    // S' beyond the largest double (a caller's Gaussians): the payoff is infinite, which rt_payoff64 gives for
    // d1 = -1, d2 = 1 and makes NaN of with d1 at its end (infinity times a phi of 0)
    if (q.S > 1.7976931348623157e308) {
        q.lnS = q.isig = 0.0;
        q.sig = -2.0;
    }
    return q;
}

// Romano-Touzi payoff C_BS(S', K, 1, sigma) (rBergLib/rBergomiMT.cpp:383-388, BlackScholes.cpp:22-26)
// = S' Phi(d1) - K Phi(d2).  With K phi(d2) = S' phi(d1) both tails come from one exponential and
// their Mills ratios, without the cancellation of the two normal CDFs far out of the money:
// Phi(d) = phi(d) M(-d) below 0, 1 - phi(d) M(d) above.  |d| beyond 1000 prices as 1000 (both are
// exactly the limit); a NaN (0 / 0: zero variance at the money) stays one.
__host__ __device__ __forceinline__ double rt_payoff64(const double* T, const PathRt64& q, double K, double lnK) {
    const double d1 = fma(q.lnS - lnK, q.isig, 0.5 * q.sig), d2 = d1 - q.sig;
    double x = fabs(d1), y = fabs(d2);
    x = x > 1000.0 ? 1000.0 : x;
    y = y > 1000.0 ? 1000.0 : y;
    double mx, my;
    mills_pair(x, y, mx, my);
    const double phi = 0.3989422804014327 * exp2_32(T, (-0.5 * EXP2_SCALE * x) * x);
    const bool p1 = d1 >= 0.0, p2 = d2 >= 0.0;
    const double c = (p1 ? q.S : 0.0) - (p2 ? K : 0.0);
    return fma(q.S * phi, (p2 ? my : -my) - (p1 ? mx : -mx), c);
}

#if defined(__HIPCC__)
// the tables into LDS (a barrier must follow before they are read)
__device__ __forceinline__ void load_exp2_tab(double* T, int tid, int nthreads) {
    for (int i = tid; i < EXP2_N; i += nthreads) T[i] = EXP2_TAB[i];
}
__device__ __forceinline__ void load_log_tab(double2* T, int tid, int nthreads) {
    double* t = reinterpret_cast<double*>(T);
    for (int i = tid; i < 2 * LOG_N; i += nthreads) t[i] = LOG_TAB[i];
}
#endif

}  // namespace rb
