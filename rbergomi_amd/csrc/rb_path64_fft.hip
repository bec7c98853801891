// rb_path64_fft.hip -- the FP64 path in one pass for longer paths: the work of k_path64
// (rb_path64.hip) with the convolution by an FP64 transform in LDS.
//
// TP = L / 16 threads own a pair of paths, L = 2^LOG2L >= 2 N:
//   1. W1, W1perp (and Wperp for plain MC) of the thread's two quads of steps of both paths, Philox
//      and Box-Muller in place or the caller's values (genGaussianMT, rBergLib/rBergomiMT.cpp:
//      169-172), kept in registers; z = W1_a + i W1_b in LDS.
//   2. Per unit (distinct H): transform, product with the transform of (a, Gamma_1, ...) / L,
//      transform back: Gamma is real, so the real and imaginary parts are the two paths' Y
//      (updateWtilde's FFTW convolution, :83-109).  x = Y + b W1perp for the thread's steps.
//   3. Per group the integrands 2^((c1 x - al P) / 32) and their sums as in k_path64.
//   4. Sums over the pair's threads (butterflies that halve the values with the lanes), to
//      ints[group][path].
//
// What bounds it: FP64 vector issue; per pair and 64 steps about 330 instructions of Gaussians, 70 of
// each group and 45 log2 L of the transforms (six-FMA butterflies, rb_fft64.h), where the
// triangular product on the matrix cores (which keep the vector unit) takes N / 2.  A thread's 16
// points and 16 steps of each stream fill the registers of two waves per SIMD (4 to 26 spilled for
// plain MC, none or 4 for Romano-Touzi; with the passes' twiddles hoisted out of the loop over the jobs
// 40 to 100, and N = 512 took 1.19 ms per 1.6e8 path steps where it then took 1.08, N = 4096 2.23 and 1.72),
// and its 17 KB of LDS per wave the CU's.  N = 2048, M = 16384, one maturity: 3.05 (k_normals,
// k_volterra_mfma_long, k_scan) -> 0.27 ms; 1.3e11 paths*steps/s at N = 1024 and 2048.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rb_fft64.h"
#include "rb_fft_lds.h"
#include "rb_kernels.h"
#include "rb_lanes.h"
#include "rb_math64.h"
#include "rb_path64.h"

namespace rb {

// ---------------------------------------------------------------- tables
__device__ __forceinline__ double2 cis_pi(double f) {  // e^(i pi f)
    double s, c;
    sincospi(f, &s, &c);
    return make_double2(c, s);
}

template <int LOG2L>
__global__ void k_fft64_twiddles(double2* __restrict__ tab) {
    using F = Fft64<LOG2L>;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F::TABLE) return;
    // forward (pass 1 ..): slot s of group J: stage r, even block b
    for (int p = 1; p <= F::PASSES; ++p) {
        const bool mid = p == F::PASSES;
        const int nj = mid ? F::TP : 1 << (4 * p), off = mid ? F::mid_off() : F::fwd_off(p);
        if (i < off || i >= off + 8 * nj) continue;
        const int s = (i - off) / nj, J = (i - off) % nj;
        const int r = s == 0 ? 3 : s == 1 ? 2 : s < 4 ? 1 : 0;
        const int b = r >= 2 ? 0 : r == 1 ? 2 * (s - 2) : 2 * (s - 4);
        const int d = LOG2L - 1 - (mid ? 0 : F::sb(p)) - r;  // 2^d blocks in the stage
        const unsigned blk = (unsigned(J) << (3 - r)) + unsigned(b);
        const double f = d > 0 ? double(__brev(blk) >> (32 - d)) / double(1 << d) : 0.0;
        tab[i] = cis_pi(-f);
    }
    for (int p = F::PASSES - 1; p >= 0; --p) {
        const int SB = F::sb(p), off = F::inv_off(p);
        if (i < off || i >= off + (8 << SB)) continue;
        const int s = (i - off) >> SB, pos = (i - off) & ((1 << SB) - 1);
        const int r = s == 0 ? 0 : s == 1 ? 1 : s < 4 ? 2 : 3;
        const int m = r <= 1 ? 0 : r == 2 ? s - 2 : s - 4;
        tab[i] = cis_pi(double(pos + (m << SB)) / double(1 << (SB + r)));
    }
}

// The spectrum of (gamma_0 .. gamma_{N-1}) / L of every unit, in the middle pass's register order:
// element 16 t + k at [k][t].  Grid: units; block TP threads.
template <int LOG2L>
__global__ void __launch_bounds__(Fft64<LOG2L>::TP) k_fft64_spectrum(const double* __restrict__ gamma, int N, int tlen,
                                                                      const double2* __restrict__ tab,
                                                                      double2* __restrict__ ghat) {
    using F = Fft64<LOG2L>;
    extern __shared__ double2 lds[];
    const int t = threadIdx.x;
    const double* g = gamma + long(blockIdx.x) * tlen;
    for (int i = t; i < F::L / 2; i += F::TP) lds[fpad64(i)] = make_double2(i < N ? g[i] : 0.0, 0.0);
    const Fft64Run<LOG2L, BlockSync> fft{lds, tab, t, BlockSync()};
    double2 x[16];
    fft.forward(x);
    constexpr double s = 1.0 / F::L;
#pragma unroll
    for (int k = 0; k < 16; ++k)
        ghat[(long(blockIdx.x) * 16 + k) * F::TP + t] = make_double2(x[k].x * s, x[k].y * s);
}

// The same unscaled and rounded to FP32, in the order of FftSpectrum, for the mixed-precision kernel
// (rb_fused_fft.hip)
template <int LOG2L>
__global__ void __launch_bounds__(Fft64<LOG2L>::TP) k_fft64_spectrum_f32(const double* __restrict__ gamma, int N,
                                                                          int tlen, const double2* __restrict__ tab,
                                                                          float2* __restrict__ ghat) {
    using F = Fft64<LOG2L>;
    extern __shared__ double2 lds[];
    const int t = threadIdx.x;
    const double* g = gamma + long(blockIdx.x) * tlen;
    for (int i = t; i < F::L / 2; i += F::TP) lds[fpad64(i)] = make_double2(i < N ? g[i] : 0.0, 0.0);
    const Fft64Run<LOG2L, BlockSync> fft{lds, tab, t, BlockSync()};
    double2 x[16];
    fft.forward(x);
#pragma unroll
    for (int k = 0; k < 16; ++k)
        ghat[long(blockIdx.x) * F::L + fft_spectrum_slot(LOG2L, 16 * t + k)] = make_float2(float(x[k].x), float(x[k].y));
}

// ---------------------------------------------------------------- the path kernel
template <int LOG2L>
struct Path64Fft {
    using F = Fft64<LOG2L>;
    static constexpr int TP = F::TP, NT = TP < 256 ? 256 : TP, PAIRS = NT / TP;
    static constexpr int W = TP < 64 ? TP : 64, NW = TP / W;  // lanes and waves of a pair
    static constexpr int EDGES = 2 * NW + 1;                  // W-quad blocks of a pair, and the end
};

// LDS behind the transforms' slots, in doubles
constexpr int P64F_MAXV = 8;  // values summed per group and pair

template <int SRC>
__device__ __forceinline__ void path64f_gauss(const Path64Args& A, const double2* lg, long p, int s, int q, double z[4]) {
    if constexpr (SRC == P64_PHILOX) {
        normals4_f64(lg, A.key, uint64_t(A.p0 + p), uint32_t(s), uint32_t(q), z);
    } else {
        const double* src = A.Z + p * A.zstride + long(s) * A.N;
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = (p < A.np && 4 * q + j < A.N) ? src[4 * q + j] : 0.0;
    }
}

// Grid (ceil(pairs / PAIRS), nsplit), block NT, dynamic LDS path64_fft_lds_bytes.
template <int LOG2L, int SRC, bool MC, int SIGNS>
__global__ void __launch_bounds__((Path64Fft<LOG2L>::NT), 2) k_path64_fft(Path64Args A) {
    using F = Fft64<LOG2L>;
    using C = Path64Fft<LOG2L>;
    using Sync = std::conditional_t<C::TP <= 64, WaveSync, BlockSync>;
    constexpr int TP = C::TP, L = F::L;
    constexpr int NV = (MC ? 3 : 2) * SIGNS, V = 2 * NV <= 4 ? 4 : 8;  // sums per path; values per group
    extern __shared__ double2 lds[];
    double2* lg = lds;                                                  // LOG_N
    double* e2 = reinterpret_cast<double*>(lds + LOG_N);                // EXP2_N
    double* red = e2 + EXP2_N;                                          // [PAIRS][NW][V]
    double2* edge = reinterpret_cast<double2*>(red + C::PAIRS * C::NW * P64F_MAXV);  // [PAIRS][2][EDGES]: W1, Wperp
    const int tid = threadIdx.x, lane = tid & 63, pair = tid / TP, t = tid % TP;
    double2* z = edge + C::PAIRS * 2 * C::EDGES + pair * F::SLOTS;
    double2* E = edge + pair * 2 * C::EDGES;
    red += pair * C::NW * P64F_MAXV;
    const Sync sync{};
    load_exp2_tab(e2, tid, C::NT);
    if constexpr (SRC == P64_PHILOX) load_log_tab(lg, tid, C::NT);
    __syncthreads();

    const int N = A.N, nq = (N + 3) >> 2;
    const long pr = long(blockIdx.x) * C::PAIRS + pair, pa = 2 * pr;
    // ---- 1. Gaussians.  At two waves per SIMD a quad's chains of dependent FP64 instructions (a logarithm,
    // a root, a sine) leave the unit idle unless other quads' fill the waits: Romano-Touzi forms the
    // quads of both paths and both streams together (N = 256, M = 655360: one quad at a time 1155 us a call, two
    // paths' 1093, all four 1051; five groups at N = 512, M = 2^19: 2891, 2820, 2713).  Plain MC has no registers
    // for the values: its loops are rolled and the values go through LDS, W1 in place for the transform, the
    // other streams through the upper half, or 16 to 60 registers are spilled (five groups at N = 512, M = 2^22: a quad at a
    // time 27.4 ms, two 26.8, the first two streams together 26.5).
    double2 w1[2][4], wp[2][4], w2[MC ? 2 : 1][4];
    if constexpr (MC) {
        auto put = [&](int at, int j, const double2(&v)[4]) {
#pragma unroll
            for (int r = 0; r < 4; ++r) z[fpad64(at + 4 * (t + TP * j) + r)] = v[r];
        };
        auto get = [&](int at, double2(&w)[2][4]) {
            WaveSync()();  // the thread's own values
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) w[j][r] = z[fpad64(at + 4 * (t + TP * j) + r)];
            WaveSync()();
        };
#pragma unroll 1
        for (int j = 0; j < 2; ++j) {
            const int q = t + TP * j;
            double g[4][4] = {};
            if (q < nq)
#pragma unroll
                for (int k = 0; k < 4; ++k) path64f_gauss<SRC>(A, lg, pa + (k & 1), k >> 1, q, g[k]);
            double2 v[4], u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = make_double2(g[0][r], g[1][r]);
                u[r] = make_double2(g[2][r], g[3][r]);
            }
            put(0, j, v);
            put(L / 2, j, u);
        }
        get(0, w1);
        get(L / 2, wp);
#pragma unroll 1
        for (int j = 0; j < 2; ++j) {
            const int q = t + TP * j;
            double g[2][4] = {};
            if (q < nq)
#pragma unroll
                for (int k = 0; k < 2; ++k) path64f_gauss<SRC>(A, lg, pa + k, 2, q, g[k]);
            double2 v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = make_double2(g[0][r], g[1][r]);
            put(L / 2, j, v);
        }
        get(L / 2, w2);
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = t + TP * j;
            double g[4][4] = {};
            if (q < nq)
#pragma unroll
                for (int k = 0; k < 4; ++k) path64f_gauss<SRC>(A, lg, pa + (k & 1), k >> 1, q, g[k]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                w1[j][r] = z[fpad64(4 * q + r)] = make_double2(g[0][r], g[1][r]);
                wp[j][r] = make_double2(g[2][r], g[3][r]);
            }
        }
    }
    // the first value of the next quad of each of the thread's quads
#pragma unroll
    for (int j = 0; j < 2; ++j)
        if (t % C::W == 0) {
            E[(t + TP * j) / C::W] = w1[j][0];
            if constexpr (MC) E[C::EDGES + (t + TP * j) / C::W] = w2[j][0];
        }
    if (t == 0) E[2 * C::NW] = E[C::EDGES + 2 * C::NW] = make_double2(0.0, 0.0);
    sync();
    bool direct = false;  // by the direct sum: a caller's W1 beyond P64_WILD in the workgroup
    if constexpr (SRC == P64_CALLER) {
        bool wild = false;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) wild |= !(fabs(w1[j][r].x) <= P64_WILD && fabs(w1[j][r].y) <= P64_WILD);
        direct = __syncthreads_or(wild);
    }
    double2 n1[2], n2[MC ? 2 : 1];
    auto next = [&](const double2(&w)[2][4], int at, double2* n) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const double2 e = E[at + (t + TP * j) / C::W + 1];
            const double sx = __shfl_down(w[j][0].x, 1, 64), sy = __shfl_down(w[j][0].y, 1, 64);
            n[j] = t % C::W == C::W - 1 ? e : make_double2(sx, sy);
        }
    };
    next(w1, 0, n1);
    if constexpr (MC) next(w2, C::EDGES, n2);

    const int j0 = int(long(A.njobs) * blockIdx.y / A.nsplit), j1 = int(long(A.njobs) * (blockIdx.y + 1) / A.nsplit);
    for (int jj = j0; jj < j1; ++jj) {
        const Path64Job job = A.jobs[jj];
        // ---- 2. x of the thread's steps
        if (jj > j0) {
            sync();  // the last job's reads are done
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) z[fpad64(4 * (t + TP * j) + r)] = w1[j][r];
        }
        // the twiddles' address is hidden from the loop over the jobs: hoisted out of it, every pass's
        // twiddles would stay in registers (40 to 100 spilled)
        int hide = 0;
        asm volatile("" : "+s"(hide));
        const double2* tw = A.tw + hide;
        const Fft64Run<LOG2L, Sync> fft{z, tw, t, sync};
        if (SRC == P64_CALLER && direct) {
            sync();
            const double* gam = A.gamma + long(job.unit) * A.tlen;
#pragma unroll 1
            for (int e = 0; e < 8; ++e) {
                const int i = 4 * (t + TP * (e >> 2)) + (e & 3);
                double2 y = make_double2(0.0, 0.0);
                for (int k = 0; k <= i && k < N; ++k) {
                    const double g = gam[k];
                    const double2 v = z[fpad64(i - k)];
                    y = make_double2(fma(g, v.x, y.x), fma(g, v.y, y.y));
                }
                z[fpad64(L / 2 + i)] = y;  // the thread's own: nothing else is read there
            }
        } else {
            double2 x[16];
            fft.forward(x);
            const double2* gh = A.ghat + long(job.unit) * L + t;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const double2 g = gh[k * TP], v = x[k];
                x[k] = make_double2(fma(-g.y, v.y, g.x * v.x), fma(g.y, v.x, g.x * v.y));
            }
            fft.backward(x);
        }
        const double b = A.units[job.unit].b;
        double2 x[2][4];
        double pj[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = t + TP * j;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double2 y = z[fpad64((SRC == P64_CALLER && direct ? L / 2 : 0) + 4 * q + r)];
                x[j][r] = make_double2(fma(b, wp[j][r].x, y.x), fma(b, wp[j][r].y, y.y));
                if constexpr (SRC == P64_CALLER) {
                    x[j][r].x = path64_caller_x(x[j][r].x, 4 * q + r < N - 1);
                    x[j][r].y = path64_caller_x(x[j][r].y, 4 * q + r < N - 1);
                }
                pj[j][r] = 4 * q + r < A.tlen ? A.ptab[long(job.unit) * A.tlen + 4 * q + r] : P64_PAD;
            }
        }
        // ---- 3. the job's groups
        for (int g = 0; g < job.gn; ++g) {
            const Path64Group& G = A.groups[job.g0 + g];
            const double c1 = G.c1, al = G.al;
            double f[V];
#pragma unroll
            for (int s = 0; s < V; ++s) f[s] = 0.0;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double ap = al * pj[j][r];
                    const double2 w = r < 3 ? w1[j][r + 1] : n1[j];
                    const double ea = exp2_32(e2, fma(c1, x[j][r].x, -ap)), eb = exp2_32(e2, fma(c1, x[j][r].y, -ap));
                    f[0] = fma(ea, ea, f[0]);
                    f[1] = fma(ea, w.x, f[1]);
                    f[NV + 0] = fma(eb, eb, f[NV + 0]);
                    f[NV + 1] = fma(eb, w.y, f[NV + 1]);
                    if constexpr (MC) {
                        const double2 v = r < 3 ? w2[j][r + 1] : n2[j];
                        f[2] = fma(ea, v.x, f[2]);
                        f[NV + 2] = fma(eb, v.y, f[NV + 2]);
                    }
                    if constexpr (SIGNS == 2) {
                        const double da = exp2_32(e2, fma(-c1, x[j][r].x, -ap)), db = exp2_32(e2, fma(-c1, x[j][r].y, -ap));
                        f[2] = fma(da, da, f[2]);
                        f[3] = fma(da, w.x, f[3]);
                        f[NV + 2] = fma(db, db, f[NV + 2]);
                        f[NV + 3] = fma(db, w.y, f[NV + 3]);
                    }
                }
            // ---- 4. sums over the pair's threads
            int idx;
            const double s = lanes_sum<C::W, V>(f, lane, idx);
            if (lane % (C::W / V) == 0) red[(t / C::W) * V + idx] = s;
            sync();
            if (t < 2 && pa + t < A.np) {
                const Path64Group Gr = G;
                double v[NV];
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    v[k] = 0.0;
                    for (int u = 0; u < C::NW; ++u) v[k] += red[u * V + t * NV + k];
                }
                // step 0: v_0 = xi
                const double w0 = t ? E[0].y : E[0].x;
                double* out = A.ints + (long(Gr.out) * A.np + pa + t) * 2;
                const double Iv = Gr.dt * (Gr.xi * (1.0 + v[0]));
                const double Is = Gr.sdt * (Gr.sxi * (w0 + v[1]));
                if constexpr (MC) {
                    const double Ip = Gr.sdt * (Gr.sxi * ((t ? E[C::EDGES].y : E[C::EDGES].x) + v[2]));
                    out[0] = Gr.rho * Is + Gr.crho * Ip - 0.5 * Iv;
                    out[1] = 0.0;
                } else {
                    out[0] = Iv;
                    out[1] = Is;
                    if constexpr (SIGNS == 2) {
                        double* o2 = A.ints2 + (long(Gr.out) * A.np + pa + t) * 2;
                        o2[0] = Gr.dt * (Gr.xi * (1.0 + v[2]));
                        o2[1] = -(Gr.sdt * (Gr.sxi * (w0 + v[3])));
                    }
                }
            }
            sync();  // red may be written again
        }
    }
}

// ---------------------------------------------------------------- host side
int path64_fft_log2(int N) {
    int l = PATH64_FFT_MIN_LOG2;
    while ((1 << l) < 2 * N) ++l;
    return l;
}

// Time of 8e7 paths*steps in microseconds, of the transforms and of the products on the matrix cores, as
// fitted to plans of 104 <= N <= 512: Gaussians, then per unit a transform (the same for every N of a length)
// or a product (growing with N), then per group.  Measured, transforms against products: Romano-Touzi, one
// unit and group at N = 224, 256, 304, 360, 384: 627, 559, 904, 771, 727 against 613, 628, 707, 808, 842; one
// unit, five groups at 256, 384: 788, 1042 against 864, 1029; three units at 176, 200, 256, 304, 336: 1607, 1420,
// 1126, 1894, 1718 against 1304, 1565, 1596, 1879, 2000; plain MC, one unit at 224, 256, 384: 831, 731, 942
// against 721, 768, 971.  Since Romano-Touzi's transforms form four quads of Gaussians together they take 48 r
// less (r: padded over real length); whole calls at N = 224, 360: 619, 759 against 627, 836, three groups at 360 934
// against 991, five at 380 1012 against 1067.  The constants are Philox plans'; with the Gaussians read from memory (8e6
// paths*steps, N from 104 to 384, one and three units, one to nine groups, both estimators) the choice is the faster kernel
// in 94 of 104 plans and within 7% of it in the rest (one unit and group, N = 208, 224, 240, 336, 384: transforms 83,
// 76, 74, 102, 93 us against 71, 74, 79, 95, 106).  Beyond N = 384 products lose even where transforms fill their
// length least (N = 400, plain MC, five groups: 1548 against 1350).
bool path64_uses_fft(int N, int units, int groups, bool mc) {
    if (N > PATH64_MFMA_MAX_N) return true;
    const double u = units, g = groups, r = double(1 << path64_fft_log2(N)) / 2 / N;
    const double fft = r * (mc ? 386 + 262 * u + 83 * g : 228 + 226 * u + 57 * g);
    const double mm = (mc ? 225 : 115) + u * (110 + 1.37 * N) + 60 * g;
    return fft < mm;
}

template <class Fn>
static hipError_t with_log2(int l, Fn fn) {
    switch (l) {
        case 9: return fn(std::integral_constant<int, 9>());
        case 10: return fn(std::integral_constant<int, 10>());
        case 11: return fn(std::integral_constant<int, 11>());
        case 12: return fn(std::integral_constant<int, 12>());
        case 13: return fn(std::integral_constant<int, 13>());
        default: return hipErrorInvalidValue;
    }
}

// as many workgroups per tile of pairs as bring four to every CU
void path64_fft_shape(Path64Args& a, int cus) {
    long tiles = 1;
    (void)with_log2(path64_fft_log2(a.N), [&](auto l) {
        constexpr int per = 2 * Path64Fft<decltype(l)::value>::PAIRS;
        tiles = (a.np + per - 1) / per;
        return hipSuccess;
    });
    const long want = (4L * cus + tiles - 1) / tiles;
    a.nsplit = int(want < a.njobs ? want : a.njobs);
}

long path64_fft_max_paths(int N) {
    long n = 0;
    (void)with_log2(path64_fft_log2(N), [&](auto l) {
        using C = Path64Fft<decltype(l)::value>;
        n = ((1L << 32) - 1) / C::NT * 2 * C::PAIRS;
        return hipSuccess;
    });
    return n;
}

size_t path64_fft_table(int N) {
    size_t n = 0;
    (void)with_log2(path64_fft_log2(N), [&](auto l) {
        n = Fft64<decltype(l)::value>::TABLE;
        return hipSuccess;
    });
    return n;
}

size_t path64_fft_lds_bytes(int N) {
    size_t n = 0;
    (void)with_log2(path64_fft_log2(N), [&](auto l) {
        using C = Path64Fft<decltype(l)::value>;
        using F = Fft64<decltype(l)::value>;
        n = (LOG_N + size_t(C::PAIRS) * (2 * C::EDGES + F::SLOTS)) * sizeof(double2) +
            (EXP2_N + size_t(C::PAIRS) * C::NW * P64F_MAXV) * sizeof(double);
        return hipSuccess;
    });
    return n;
}

hipError_t launch_path64_fft_tables(const double* gamma, int nunits, int N, int tlen, double2* tw, double2* ghat,
                                    hipStream_t st) {
    return with_log2(path64_fft_log2(N), [&](auto l) -> hipError_t {
        constexpr int LOG2L = decltype(l)::value;
        using F = Fft64<LOG2L>;
        const size_t lds = F::SLOTS * sizeof(double2);
        if (lds > 65536) {
            const hipError_t e = allow_lds(reinterpret_cast<const void*>(&k_fft64_spectrum<LOG2L>), lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL((k_fft64_twiddles<LOG2L>), dim3((F::TABLE + 255) / 256), dim3(256), 0, st, tw);
        hipLaunchKernelGGL((k_fft64_spectrum<LOG2L>), dim3(unsigned(nunits)), dim3(F::TP), lds, st, gamma, N, tlen, tw,
                           ghat);
        return hipGetLastError();
    });
}

hipError_t launch_fft_spectrum_f32(const double* gamma, int nunits, int N, int tlen, int log2L, double2* tw,
                                   float2* ghat, hipStream_t st) {
    return with_log2(log2L, [&](auto l) -> hipError_t {
        constexpr int LOG2L = decltype(l)::value;
        using F = Fft64<LOG2L>;
        const size_t lds = F::SLOTS * sizeof(double2);
        if (lds > 65536) {
            const hipError_t e = allow_lds(reinterpret_cast<const void*>(&k_fft64_spectrum_f32<LOG2L>), lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL((k_fft64_twiddles<LOG2L>), dim3((F::TABLE + 255) / 256), dim3(256), 0, st, tw);
        hipLaunchKernelGGL((k_fft64_spectrum_f32<LOG2L>), dim3(unsigned(nunits)), dim3(F::TP), lds, st, gamma, N, tlen,
                           tw, ghat);
        return hipGetLastError();
    });
}

hipError_t launch_path64_fft(const Path64Args& a, hipStream_t st) {
    if (a.np < 1 || a.njobs < 1 || a.nsplit < 1 || a.N > PATH64_FFT_MAX_N || a.np > path64_fft_max_paths(a.N))
        return hipErrorInvalidValue;
    return with_log2(path64_fft_log2(a.N), [&](auto l) -> hipError_t {
        constexpr int LOG2L = decltype(l)::value;
        using C = Path64Fft<LOG2L>;
        const size_t lds = path64_fft_lds_bytes(a.N);
        const long pairs = (a.np + 1) / 2;
        const dim3 grid(unsigned((pairs + C::PAIRS - 1) / C::PAIRS), unsigned(a.nsplit));
        auto go = [&](auto kern) -> hipError_t {
            if (lds > 65536) {
                const hipError_t e = allow_lds(reinterpret_cast<const void*>(kern), lds);
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL(kern, grid, dim3(C::NT), lds, st, a);
            return hipGetLastError();
        };
        if (a.signs == 2)
            return a.src != P64_PHILOX || a.mc ? hipErrorInvalidValue : go(&k_path64_fft<LOG2L, P64_PHILOX, false, 2>);
        auto from = [&](auto src) {
            constexpr int SRC = decltype(src)::value;
            return a.mc ? go(&k_path64_fft<LOG2L, SRC, true, 1>) : go(&k_path64_fft<LOG2L, SRC, false, 1>);
        };
        switch (a.src) {
            case P64_PHILOX: return from(std::integral_constant<int, P64_PHILOX>());
            case P64_MEMORY: return from(std::integral_constant<int, P64_MEMORY>());
            case P64_CALLER: return from(std::integral_constant<int, P64_CALLER>());
            default: return hipErrorInvalidValue;
        }
    });
}

}  // namespace rb
