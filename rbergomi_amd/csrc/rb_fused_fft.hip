// rb_fused_fft.hip -- mixed-precision pricing by FFT convolution in one pass over the paths: for long
// paths (N > 1024, where the Toeplitz GEMM's W1 tile no longer fits LDS), and for any N <= 8192 at the
// FFT precision.
//
// TP threads own a pair of paths, half of them each path: TP = L / 16 (512 at L = 2^14), L = 2^LOG2L >= 2 N:
//   1. W1 of the thread's quads of steps of its path, Philox and FP32 Box-Muller (genGaussianMT,
//      rBergLib/rBergomiMT.cpp:169-172), kept in registers.
//   2. Per unit (distinct H): z = W1_a + i W1_b through the LDS transforms (rb_fft_lds.h, natural order),
//      with the product by the spectrum of (a, Gamma_1, ..., Gamma_{N-1}) between them: Gamma is real, so the
//      real and imaginary parts are the two paths' convolutions (updateWtilde's FFTW convolution,
//      :83-109).  Wtilde = sc (Y + b W1perp) for the thread's steps.
//   3. Per (H, eta, T) group sqrt(v_i) = exp2(c1 Wtilde_{i-1} - al P_i - be) and the sums of v and
//      sqrt(v) W1 in FP32 over up to eight quads of steps, then in FP64 (scaleWtilde/updateV/intVdt/
//      intRootVdW, :73-80, 163-167, 427-436); plain MC adds sqrt(v) Wperp.  P = +inf at i = 0 and i >= N
//      makes those terms exactly 0.
//   4. ints[group][path]: the integrals (Iv, Is[, Ip]) in FP64, priced by the payoff kernel of
//      rb_payoff64.hip in chunks of paths.
//
// What bounds it: vector issue (per thread of 16 steps and unit about 900 instructions of Gaussians, 1500 of
// butterflies, 100 of each group; 61% of N = 4096's time below at the measured issue costs).  Sixteen points per thread keep
// four waves per SIMD in registers (no spills to N = 2048, 17 to 4096, plain MC 25) and LDS (9 KB a wave); at N > 4096,
// where one workgroup fills the LDS, two waves of thirty-two points each.  The form before it, one
// pair per 256 threads with the payoffs of both paths priced between barriers by one thread per option
// and the tables formed on the host, took, one maturity, N = 4096, M = 32768, 1.02 ms (now 0.67), N =
// 2048, M = 65536 1.02 (0.53), plain MC 1.56 and 1.09 (0.74 and 0.53), N = 512, M = 200000 1.61 (0.34), and
// its tables 1.3 ms of each request at N = 4096.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rb_fft_lds.h"
#include "rb_fused.h"
#include "rb_kernels.h"
#include "rb_lanes.h"

namespace rb {

// ---------------------------------------------------------------- tables
// k^h to the nearest double, through a logarithm and an exponential of twice its length: the error of
// a library power, 1e-12 in the spectrum of its differences, turns a rounding of the FP32 spectrum in one
// request of two and moves its prices by 5e-10.
struct Dd {
    double hi, lo;
};
__device__ inline Dd dd_norm(double a, double b) {  // |a| >= |b|
#pragma clang fp contract(off)
    const double s = a + b;
    return Dd{s, b - (s - a)};
}
__device__ inline Dd dd_mul(Dd a, Dd b) {
#pragma clang fp contract(off)
    const double p = a.hi * b.hi;
    return dd_norm(p, fma(a.hi, b.hi, -p) + fma(a.hi, b.lo, a.lo * b.hi));
}
__device__ inline Dd dd_exp(Dd x) {  // 2^n (Taylor series of the rest over 64)^64
#pragma clang fp contract(off)
    constexpr double LN2_HI = 0.693147180559945286, LN2_LO = 2.31904681384629956e-17;
    const double n = rint(x.hi / LN2_HI), p = n * LN2_HI;
    const Dd d = dd_norm(x.hi - p, (x.lo - fma(n, LN2_HI, -p)) - n * LN2_LO);
    const Dd r{d.hi * 0x1p-6, d.lo * 0x1p-6};
    Dd e{1.0, 0.0};
    for (int k = 9; k >= 1; --k) {  // 1 + r e / k
        e = dd_mul(r, e);
        const double q = e.hi / k;
        e = dd_norm(q, (fma(-q, double(k), e.hi) + e.lo) / k);
        const double s = 1.0 + e.hi;
        e = dd_norm(s, (e.hi - (s - 1.0)) + e.lo);
    }
    for (int k = 0; k < 6; ++k) e = dd_mul(e, e);
    return Dd{ldexp(e.hi, int(n)), ldexp(e.lo, int(n))};
}
__device__ inline double pow_nearest(double k, double h) {
#pragma clang fp contract(off)
    const double l = log(k);
    const Dd e = dd_exp(Dd{-l, 0.0});
    const Dd t = dd_mul(dd_norm(l, fma(k, e.hi, -1.0) + k * e.lo), Dd{h, 0.0});
    return dd_exp(t).hi;
}

// gamma[u][i]: a, Gamma_1 .. Gamma_{N-1}; ptab[u][i] = P_i, +inf at 0 and from N on
__global__ void k_fft32_tables(const Unit* __restrict__ units, int N, int tlen, double off, double* __restrict__ gamma,
                               float* __restrict__ ptab) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= tlen) return;
    const Unit un = units[blockIdx.y];
    const double h = un.H - 0.5 + 1.0;
    double g = 0.0;
    if (i == 0) g = un.a;
    else if (i < N && gamma) g = (pow_nearest(i + 1.0, h) - pow_nearest(double(i), h)) / h;
    if (gamma) gamma[long(blockIdx.y) * tlen + i] = g;
    ptab[long(blockIdx.y) * tlen + i] = i >= 1 && i < N ? float(pow(double(i) - off, 2.0 * un.H)) : INFINITY;
}

// Twiddles: exp(-2 pi i k / L) for k < L/2, then the passes' tables (FftPassTable)
__global__ void k_fft32_twiddles(int log2L, float2* __restrict__ tw) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, H2 = 1 << (log2L - 1);
    if (i >= fused_fft_table(log2L)) return;
    double s, c;
    sincospi(-double(fft_twiddle_power(log2L, i)) / double(H2), &s, &c);
    tw[i] = make_float2(float(c), float(s));
}

// ---------------------------------------------------------------- the path kernel
template <int LOG2L>
struct FftPair {
    static constexpr int L = 1 << LOG2L;
    static constexpr int TP = LOG2L <= 13 ? L / 16 : 512, HP = TP / 2;  // threads of a pair, of a path
    static constexpr int NT = TP < 256 ? 256 : TP, PAIRS = NT / TP;
    static constexpr int W = HP < 64 ? HP : 64, NW = HP / W;  // lanes and waves of a path
    static constexpr int QT = L / 8 / HP;                     // quads of steps per thread
    // A path's sums run in FP32 over the quads q, q + 256, ... (CQ of them), then in FP64
    static constexpr int CQ = LOG2L <= 11 ? 1 : 1 << (LOG2L - 11);
    // element i in slot i + i / 16: the accesses of every pass spread over the banks (i / 32, half of them
    // two lanes to a bank)
    static constexpr int PAD = 4, SLOTS = L + (L >> PAD);
    __device__ static __forceinline__ int slot(int i) { return i + (i >> PAD); }
    __device__ static __forceinline__ int quad(int s, int j) { return s + HP * (j / CQ) + 256 * (j % CQ); }
    // waves per SIMD the registers are cut for
    static constexpr int WAVES = LOG2L <= 13 ? 4 : 2;
};

// A pass of the transform by the TP threads of a pair (the schedules of rb_fft_lds.h)
template <int TP, class Sync>
struct FftPairPass {
    int t;
    Sync sync;
    template <int LOG2L, int SB, int R, int KIND, class GT>
    __device__ __forceinline__ void pass(float2* z, FftPassTable tw, GT G) const {
        constexpr int NG = (1 << LOG2L) >> R;
        static_assert(NG % TP == 0, "whole groups per thread");
#pragma unroll 2
        for (int u = 0; u < NG / TP; ++u) fft_group<LOG2L, SB, R, KIND, FftPair<LOG2L>::PAD>(z, tw, G, t + TP * u);
        sync();
    }
};

// The first pass of the forward transform by the TP threads of a pair (fft_first_load and what follows)
template <int LOG2L, int TP, class Sync>
__device__ __forceinline__ void fft_first_pass(float2* z, const float2* tw, int t, const Sync& sync) {
    constexpr int span = 1 << (LOG2L - 5), PAD = FftPair<LOG2L>::PAD;
    const int pos = t & (span - 1);
    float2 x[16];
    fft_first_load<LOG2L, PAD>(x, z, pos);
    if constexpr (TP == 2 * span) {  // half of the threads to each half of the points
        sync();                      // the lower half has been read
        if (t >= span) fft_first_upper<LOG2L>(x, tw, pos);
        fft_first_store<LOG2L, PAD>(x, z, tw, pos, t >= span ? 1 : 0);
    } else {
        static_assert(TP == span, "both halves of a group to a thread");
        float2 y[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) y[k] = x[k];
        fft_first_store<LOG2L, PAD>(x, z, tw, pos, 0);
        fft_first_upper<LOG2L>(y, tw, pos);
        fft_first_store<LOG2L, PAD>(y, z, tw, pos, 1);
    }
    sync();
}

// Grid (ceil(pairs / PAIRS), nsplit), block NT, dynamic LDS fused_fft_lds.
template <int LOG2L, bool MC>
__global__ void __launch_bounds__((FftPair<LOG2L>::NT), (FftPair<LOG2L>::WAVES)) k_fused_fft(FftFusedArgs A) {
    using C = FftPair<LOG2L>;
    using Sync = std::conditional_t<C::TP <= 64, WaveSync, BlockSync>;
    constexpr int TP = C::TP, HP = C::HP, QT = C::QT, CQ = C::CQ, L = C::L, H2 = L / 2;
    constexpr int NV = MC ? 3 : 2, V = MC ? 4 : 2;  // sums per path; values summed over the lanes
    extern __shared__ double2 lds[];
    double* red = reinterpret_cast<double*>(lds);  // [PAIRS][2][NW][V]
    const int tid = threadIdx.x, lane = tid & 63, pair = tid / TP, t0 = tid % TP;
    const int c = t0 / HP, s0 = t0 % HP;  // the thread's path of the pair
    float2* z = reinterpret_cast<float2*>(red + C::PAIRS * 2 * C::NW * V) + pair * (C::SLOTS + L / 8);
    float* last = reinterpret_cast<float*>(z + C::SLOTS) + c * (L / 8);  // [quads]: Wtilde of a quad's last step
    red += (pair * 2 + c) * C::NW * V;
    const Sync sync{};
    const int N = A.N, nq = (N + 3) >> 2;
    const long pr = long(blockIdx.x) * C::PAIRS + pair, p = 2 * pr + c;
    // ---- 1. Gaussians of the thread's quads, two at a time where the whole wave needs both: their chains of
    // dependent instructions fill each other's waits (one at a time, N = 4096, M = 32768: 698 us a call, now 689;
    // N = 2048, M = 60003, two maturities 551 -> 544; drawn for lanes that need one only, N = 1100 lost 3%)
    auto gaussians = [&](uint32_t stream, int s, float(&w)[QT][4]) {
#pragma unroll
        for (int j = 0; j < QT; j += 2) {
            const int q = C::quad(s, j), qn = C::quad(s, j + 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) w[j][r] = w[j + 1][r] = 0.f;
            if (__all(qn < nq)) {
                normals4_f32(A.key, uint64_t(A.p0 + p), stream, uint32_t(q), w[j]);
                normals4_f32(A.key, uint64_t(A.p0 + p), stream, uint32_t(qn), w[j + 1]);
            } else {
                if (q < nq) normals4_f32(A.key, uint64_t(A.p0 + p), stream, uint32_t(q), w[j]);
                if (qn < nq) normals4_f32(A.key, uint64_t(A.p0 + p), stream, uint32_t(qn), w[j + 1]);
            }
        }
    };
    float w1[QT][4];
    gaussians(0, s0, w1);
#pragma unroll
    for (int j = 0; j < QT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * C::quad(s0, j) + r >= N) w1[j][r] = 0.f;

    const int u0 = int(long(A.nunits) * blockIdx.y / A.nsplit), u1 = int(long(A.nunits) * (blockIdx.y + 1) / A.nsplit);
    for (int u = u0; u < u1; ++u) {
        const FusedUnit U = A.units[u];
        // the thread's place and the tables' address are hidden from the loop over the units: hoisted out
        // of it, every pass's addresses and twiddles would stay in registers (60 to 100 spilled)
        int t = t0, s = s0, hide = 0;
        asm volatile("" : "+v"(t), "+v"(s), "+s"(hide));
        const float2* tw = A.tw + hide;
        // ---- 2. Wtilde of the thread's steps
        if (u > u0) sync();  // the last unit's reads are done
#pragma unroll
        for (int j = 0; j < QT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) reinterpret_cast<float*>(z + C::slot(4 * C::quad(s, j) + r))[c] = w1[j][r];
        sync();
        fft_first_pass<LOG2L, TP>(z, tw, t, sync);
        fft_nat_fwd<LOG2L, LOG2L - 6>(z, FftPassTable{tw + H2}, FftSpectrum{A.ghat + long(u) * L},
                                        FftPairPass<TP, Sync>{t, sync});
        asm volatile("" : "+v"(s));  // its slots are formed again after the transforms (24 fewer spilled)
        // W1perp is drawn here, once per unit: held across the transforms, its registers would not leave
        // four waves per SIMD
        float x[QT][4];
        gaussians(1, s, x);
        constexpr float invL = 1.0f / float(L);
        auto wtilde = [&](auto comp) {
#pragma unroll
            for (int j = 0; j < QT; ++j) {
                const int i0 = 4 * C::quad(s, j);
#pragma unroll
                for (int r = 0; r < 4; ++r) {  // the inverse top stage: z_i + conj(W_L^i) z_{i + L/2}
                    const float2 lo = z[C::slot(i0 + r)], hi = z[C::slot(i0 + r + H2)], w = tw[i0 + r];
                    const float2 m = fft_mul<FFT_MUL_Y>(hi, make_float2(w.x, -w.y));
                    const float y = decltype(comp)::value ? lo.y + m.y : lo.x + m.x;
                    x[j][r] = U.sc * fmaf(y, invL, U.b * x[j][r]);
                }
                last[C::quad(s, j)] = x[j][3];
            }
        };
        if (c == 0) wtilde(std::integral_constant<int, 0>());
        else wtilde(std::integral_constant<int, 1>());
        float w2[QT][4];
        if constexpr (MC) gaussians(2, s, w2);
        sync();
        // v_i takes Wtilde_{i-1}: the quads move up by one step
        float pj[QT][4];
#pragma unroll
        for (int j = 0; j < QT; ++j) {
            const int q = C::quad(s, j);
            const float4 p4 = *reinterpret_cast<const float4*>(A.ptab + long(u) * H2 + 4 * q);
            pj[j][0] = p4.x;
            pj[j][1] = p4.y;
            pj[j][2] = p4.z;
            pj[j][3] = p4.w;
            x[j][3] = x[j][2];
            x[j][2] = x[j][1];
            x[j][1] = x[j][0];
            x[j][0] = q > 0 ? last[q - 1] : 0.f;
        }
        // ---- 3. the unit's groups
        for (int g = U.g_begin; g < U.g_end; ++g) {
            const FusedGroup& G = A.groups[g];
            const float c1 = G.c1, al = G.al, be = G.be;
            double d[V];
#pragma unroll
            for (int k = 0; k < V; ++k) d[k] = 0.0;
#pragma unroll
            for (int j0 = 0; j0 < QT; j0 += CQ) {
                float f0 = 0.f, f1 = 0.f, f2 = 0.f;
#pragma unroll
                for (int j = j0; j < j0 + CQ; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = fmaf(al, pj[j][r], be);
                        const float sv = __builtin_amdgcn_exp2f(fmaf(x[j][r], c1, -e));
                        f0 = fmaf(sv, sv, f0);
                        f1 = fmaf(sv, w1[j][r], f1);
                        if constexpr (MC) f2 = fmaf(sv, w2[j][r], f2);
                    }
                d[0] += double(f0);
                d[1] += double(f1);
                if constexpr (MC) d[2] += double(f2);
            }
            // ---- 4. FP64 sums over the path's threads
            int idx;
            const double sum = lanes_sum<C::W, V>(d, lane, idx);
            if (lane % (C::W / V) == 0) red[(s / C::W) * V + idx] = sum;
            sync();
            if (s == 0 && p < A.np) {
                double v[NV];
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    v[k] = 0.0;
                    for (int w = 0; w < C::NW; ++w) v[k] += red[w * V + k];
                }
                // step 0: v_0 = xi
                double* out = A.ints + (long(g) * A.np + p) * NV;
                out[0] = G.dt * (G.xi + v[0]);
                out[1] = G.sdt * (G.sxi * double(w1[0][0]) + v[1]);
                if constexpr (MC) out[2] = G.sdt * (G.sxi * double(w2[0][0]) + v[2]);
            }
            sync();  // red may be written again
        }
    }
}

// ---------------------------------------------------------------- host side
int fused_fft_log2(int N) {
    int l = 10;
    while ((1 << l) < 2 * N) ++l;
    return l;
}

template <class Fn>
static hipError_t with_log2(int l, Fn fn) {
    switch (l) {
        case 10: return fn(std::integral_constant<int, 10>());
        case 11: return fn(std::integral_constant<int, 11>());
        case 12: return fn(std::integral_constant<int, 12>());
        case 13: return fn(std::integral_constant<int, 13>());
        case 14: return fn(std::integral_constant<int, 14>());
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_fused_fft_tables(const Unit* units, int nunits, int N, double off, double* gamma, double2* tw64,
                                   float* ptab, float2* tw, float2* ghat, hipStream_t st) {
    const int log2L = fused_fft_log2(N), tlen = 1 << (log2L - 1);
    hipLaunchKernelGGL(k_fft32_tables, dim3(unsigned((tlen + 63) / 64), unsigned(nunits)), dim3(64), 0, st, units, N,
                       tlen, off, gamma, ptab);
    hipLaunchKernelGGL(k_fft32_twiddles, dim3(unsigned((fused_fft_table(log2L) + 255) / 256)), dim3(256), 0, st, log2L, tw);
    if (gamma) {
        const hipError_t e = launch_fft_spectrum_f32(gamma, nunits, N, tlen, log2L, tw64, ghat, st);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

hipError_t launch_fused_fft(FftFusedArgs a, int cus, hipStream_t st) {
    if (a.np < 1 || a.N < 1 || a.N > 8192 || a.nunits < 1) return hipErrorInvalidValue;
    return with_log2(fused_fft_log2(a.N), [&](auto l) -> hipError_t {
        constexpr int LOG2L = decltype(l)::value;
        using C = FftPair<LOG2L>;
        const int V = a.mc ? 4 : 2;
        const size_t lds = size_t(C::PAIRS) * (2 * C::NW * V * sizeof(double) + (C::SLOTS + C::L / 8) * sizeof(float2));
        const long tiles = ((a.np + 1) / 2 + C::PAIRS - 1) / C::PAIRS;
        // the units of a tile over as many workgroups as bring four to every CU
        const long want = (4L * cus + tiles - 1) / tiles;
        a.nsplit = int(want < a.nunits ? want : a.nunits);
        auto go = [&](auto kern) -> hipError_t {
            if (lds > 65536) {
                const hipError_t e = allow_lds(reinterpret_cast<const void*>(kern), lds);
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL(kern, dim3(unsigned(tiles), unsigned(a.nsplit)), dim3(C::NT), lds, st, a);
            return hipGetLastError();
        };
        return a.mc ? go(&k_fused_fft<LOG2L, true>) : go(&k_fused_fft<LOG2L, false>);
    });
}

}  // namespace rb
