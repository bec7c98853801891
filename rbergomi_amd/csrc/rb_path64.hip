// rb_path64.hip -- the FP64 path in one pass: from Gaussians to the integrals of every group, with
// nothing per step in HBM (N <= 384 where products are cheaper than transforms, path64_uses_fft; rb_path64_fft.hip else).
//
// A workgroup owns a tile of 16 PT paths (PT = 1, 2 or 4 sub-tiles of 16):
//   1. W1 of the tile, k-major in LDS: Philox and Box-Muller in place (genGaussianMT,
//      rBergLib/rBergomiMT.cpp:169-172), or the caller's values from memory.
//   2. Per unit (distinct H), 16-row blocks of Y = Gamma * W1 + a W1 on v_mfma_f64_16x16x4_f64 as a
//      lower-triangular Toeplitz product (updateWtilde, :83-109), A from a zero-padded LDS copy of
//      (a, Gamma_1, ...), B from the tile.  The rows of a block are permuted so that a lane's four
//      results are four consecutive steps of one path: exactly one Philox block of W1perp.
//   3. x = Y + b W1perp in registers, then for each of the job's groups the four integrands
//      sqrt(v) = 2^((c1 x - al P) / 32) (scaleWtilde, updateV, :73-80, 163-167) and the sums of v
//      and sqrt(v) W1 (intVdt, intRootVdW, :427-436); plain MC adds sqrt(v) Wperp (updateZ,
//      updateS, :111-136).  Rows past the last step read P64_PAD and contribute exactly zero.
//   4. Sums over the tile's lanes and waves, in a fixed order, to ints[group][path].
//
// What bounds it: the issue of vector instructions.  An FP64 MFMA keeps its SIMD's vector unit for
// all of its 73 cycles (measured: waves of MFMA beside waves of FP64, FP32 or integer work take the
// sum of their times), so a product costs what its 16 FP64 FMAs would; at N = 256 the convolution
// is 42% of the kernel's time, the two Gaussian streams most of the rest.  Keeping every step on chip
// takes away 24 bytes of HBM per path, step and Gaussian stream or process of the staged kernels
// (k_normals, k_volterra_mfma, k_scan): N = 256, M = 655360, one maturity 3.17 -> 1.33 ms; N = 512,
// M = 2^19, five maturities 9.17 -> 4.89 ms; 250 distinct H on N = 200, M = 10^4 5.61 -> 3.1 ms.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rb_kernels.h"
#include "rb_math64.h"
#include "rb_mfma.h"
#include "rb_path64.h"

namespace rb {

// ---------------------------------------------------------------- tables
// Gamma_k = ((k+1)^h - k^h) / h, h = H + 1/2 (getGamma, rBergLib/rBergomiMT.cpp:143-149), as
// k^h (e^{h ln(1 + 1/k)} - 1) / h, which does not cancel; entry 0 is the first-cell weight a.
__global__ void k_path64_tables(const Unit* __restrict__ units, int N, int tlen, double off,
                                double* __restrict__ gamma, double* __restrict__ ptab) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= tlen) return;
    const Unit un = units[blockIdx.y];
    const double h = un.H + 0.5;
    double g = 0.0;
    if (i == 0) g = un.a;
    else if (i < N) g = pow(double(i), h) * expm1(h * log1p(1.0 / double(i))) / h;
    gamma[long(blockIdx.y) * tlen + i] = g;
    ptab[long(blockIdx.y) * tlen + i] = i + 1 < N ? pow(double(i + 1) - off, 2.0 * un.H) : P64_PAD;
}

hipError_t launch_path64_tables(const Unit* units, int nunits, int N, int tlen, double off, double* gamma,
                                double* ptab, hipStream_t st) {
    hipLaunchKernelGGL(k_path64_tables, dim3(unsigned((tlen + 63) / 64), unsigned(nunits)), dim3(64), 0, st, units, N,
                       tlen, off, gamma, ptab);
    return hipGetLastError();
}

// ---------------------------------------------------------------- the path kernel
constexpr size_t P64_LDS_CU = 160 * 1024;

// row blocks with a row below N - 1 (Wtilde_{N-1} is not used)
__host__ __device__ inline int path64_blocks(int N) { return (N + 14) >> 4; }
// sub-tiles of 16 paths per workgroup: as many as keep four waves on row blocks
__host__ __device__ inline int path64_subtiles(int N) {
    const int nb = path64_blocks(N);
    return nb <= 1 ? 4 : nb == 2 ? 2 : 1;
}

struct Path64Lds {
    size_t lg, e2, gs, ws, vs, w20, red, bytes;  // offsets in bytes
};

__host__ __device__ inline Path64Lds path64_lds(int tlen, int PT, int waves, int greg, bool mc, int signs, bool perp) {
    Path64Lds l;
    size_t o = 0;
    l.lg = o;
    o += LOG_N * sizeof(double2);
    l.e2 = o;
    o += EXP2_N * sizeof(double);
    l.gs = o;
    o += size_t(16 + tlen) * sizeof(double);
    l.ws = o;
    o += size_t(PT) * (tlen + 1) * 16 * sizeof(double);
    l.vs = o;
    if (perp) o += size_t(PT) * tlen * 16 * sizeof(double);
    l.w20 = o;
    if (mc) o += size_t(PT) * (tlen / 16 + 1) * 16 * sizeof(double);
    l.red = o;
    o += size_t(waves) * greg * (mc ? 3 : 2) * signs * 16 * sizeof(double);
    l.bytes = o;
    return l;
}

size_t path64_lds_bytes(const Path64Args& a) {
    return path64_lds(a.tlen, path64_subtiles(a.N), a.threads / 64, a.greg, a.mc != 0, a.signs, a.cache_perp != 0).bytes;
}

// Launch shape of a.np paths (N, tlen, njobs, greg, mc, signs given).  W1perp is kept in LDS when a
// workgroup has several jobs and two workgroups still fit a CU.  Eight waves share a tile where its
// LDS leaves a CU fewer than three workgroups: the kernel's 128 registers allow four waves per SIMD.
// The jobs are split over as many workgroups per tile as bring four workgroups to every CU.
void path64_shape(Path64Args& a, int cus) {
    const int per = 16 * path64_subtiles(a.N);
    const long tiles = (a.np + per - 1) / per;
    const long want = (4L * cus + tiles - 1) / tiles;
    a.nsplit = int(want < a.njobs ? want : a.njobs);
    a.threads = 256;
    a.cache_perp = a.njobs > a.nsplit;
    if (path64_lds_bytes(a) > P64_LDS_CU / 2) a.cache_perp = 0;
    if (path64_lds_bytes(a) > P64_LDS_CU / 3 && path64_blocks(a.N) >= 8) a.threads = 512;
}

// tiles by the larger of the two workgroup sizes
long path64_max_paths(int N) { return ((1L << 32) - 1) / 512 * 16 * path64_subtiles(N); }

// groups per job: the smallest instantiated count that holds a unit's groups, 8 at most
int path64_greg(int most, int signs) { return signs == 2 || most <= 2 ? 2 : most <= 4 ? 4 : 8; }

// four values of stream s of path p (memory index) at steps 4q .. 4q + 3
template <int SRC>
__device__ __forceinline__ void path64_gauss(const Path64Args& A, const double2* lg, long p, int s, int q, double z[4]) {
    if constexpr (SRC == P64_PHILOX) {
        normals4_f64(lg, A.key, uint64_t(A.p0 + p), uint32_t(s), uint32_t(q), z);
    } else {
        const double* src = A.Z + p * A.zstride + long(s) * A.N;
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = (p < A.np && 4 * q + j < A.N) ? src[4 * q + j] : 0.0;
    }
}

__device__ __forceinline__ double sum_kq(double v) {  // over the four lanes of a path
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// Grid (tiles, nsplit), block NT, dynamic LDS path64_lds_bytes.
template <int SRC, bool MC, int SIGNS, int GREG, int NT>
__global__ void __launch_bounds__(NT, 4) k_path64(Path64Args A) {
    extern __shared__ double2 lds[];
    constexpr int NS = (MC ? 3 : 2) * SIGNS;
    const int N = A.N, tlen = A.tlen;
    const int PT = path64_subtiles(N);
    const int nb = path64_blocks(N);
    const Path64Lds L = path64_lds(tlen, PT, NT / 64, GREG, MC, SIGNS, A.cache_perp != 0);
    char* base = reinterpret_cast<char*>(lds);
    double2* lg = reinterpret_cast<double2*>(base + L.lg);
    double* e2 = reinterpret_cast<double*>(base + L.e2);
    double* Gs = reinterpret_cast<double*>(base + L.gs);   // Gs[16 + t] = Gamma_t (a at 0), 0 below
    double* Ws = reinterpret_cast<double*>(base + L.ws);   // [PT][tlen + 1][16], W1 of step k at k
    double* Vs = reinterpret_cast<double*>(base + L.vs);   // [PT][tlen][16], W1perp (cache_perp)
    double* W20 = reinterpret_cast<double*>(base + L.w20); // [PT][tlen / 16 + 1][16], Wperp at 16 rb
    double* red = reinterpret_cast<double*>(base + L.red); // [waves][GREG][NS][16]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long pb = long(blockIdx.x) * 16 * PT;
    const int psh = PT == 1 ? 4 : PT == 2 ? 5 : 6;

    load_exp2_tab(e2, tid, NT);
    if constexpr (SRC == P64_PHILOX) {
        load_log_tab(lg, tid, NT);
        __syncthreads();
    }
    // ---- 1. the tile's Gaussians
    if (A.cache_perp) {
        // both streams of a quad together: their chains of dependent instructions fill each other's waits
        // (plain MC, N = 200, M = 100003, two H: 405 -> 396 us a call)
        for (int t = tid; t < (tlen >> 2) << psh; t += NT) {
            const int pp = t & ((1 << psh) - 1), q = t >> psh;
            double z[4], y[4];
            path64_gauss<SRC>(A, lg, pb + pp, 0, q, z);
            path64_gauss<SRC>(A, lg, pb + pp, 1, q, y);
            double* w = Ws + (size_t(pp >> 4) * (tlen + 1) + 4 * q) * 16 + (pp & 15);
            double* v = Vs + (size_t(pp >> 4) * tlen + 4 * q) * 16 + (pp & 15);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                w[16 * j] = z[j];
                v[16 * j] = y[j];
            }
        }
    } else {
        for (int t = tid; t < (tlen >> 2) << psh; t += NT) {
            const int pp = t & ((1 << psh) - 1), q = t >> psh;
            double z[4];
            path64_gauss<SRC>(A, lg, pb + pp, 0, q, z);
            double* w = Ws + (size_t(pp >> 4) * (tlen + 1) + 4 * q) * 16 + (pp & 15);
#pragma unroll
            for (int j = 0; j < 4; ++j) w[16 * j] = z[j];
        }
    }
    if (tid < 1 << psh) Ws[(size_t(tid >> 4) * (tlen + 1) + tlen) * 16 + (tid & 15)] = 0.0;
    if constexpr (MC)  // Wperp at the first step of every row block (and 0 past the last)
        for (int t = tid; t < ((tlen >> 4) + 1) << psh; t += NT) {
            const int pp = t & ((1 << psh) - 1), rb = t >> psh;
            double z[4] = {0.0, 0.0, 0.0, 0.0};
            if (16 * rb < tlen) path64_gauss<SRC>(A, lg, pb + pp, 2, 4 * rb, z);
            W20[(size_t(pp >> 4) * (tlen / 16 + 1) + rb) * 16 + (pp & 15)] = z[0];
        }

    const int KW = NT / 64 / PT;                       // waves per sub-tile
    const int sub = wave / KW, kw = wave - sub * KW;
    const int m = lane & 15, kq = lane >> 4;
    const int perm = 4 * (m & 3) + (m >> 2);     // the step of hardware row m within a block
    const double* W = Ws + size_t(sub) * (tlen + 1) * 16 + m;
    const long p = pb + 16 * sub + m;
    const int j0 = int(long(A.njobs) * blockIdx.y / A.nsplit), j1 = int(long(A.njobs) * (blockIdx.y + 1) / A.nsplit);
    for (int jj = j0; jj < j1; ++jj) {
        const Path64Job job = A.jobs[jj];
        if (jj == j0 || A.jobs[jj - 1].unit != job.unit) {
            const double* g = A.gamma + long(job.unit) * tlen;
            for (int t = tid; t < 16 + tlen; t += NT) Gs[t] = t < 16 ? 0.0 : g[t - 16];
        }
        __syncthreads();
        const double b = A.units[job.unit].b;
        const double* P = A.ptab + long(job.unit) * tlen;
        const Path64Group* G = A.groups + job.g0;
        double f[GREG][NS];
#pragma unroll
        for (int g = 0; g < GREG; ++g)
#pragma unroll
            for (int s = 0; s < NS; ++s) f[g][s] = 0.0;
        // row blocks from the longest down, dealt to the sub-tile's waves back and forth
#pragma unroll 1
        for (int j = 0; j * KW < nb; ++j) {
            const int rb = nb - 1 - (j * KW + ((j & 1) ? KW - 1 - kw : kw));
            if (rb < 0) break;
            const int i0 = 16 * rb, q = 4 * rb + kq;
            // ---- 2. Y of the block: chunk c covers steps 4c .. 4c + 3 <= i0 + 15
            const int nc = 4 * (rb + 1);
            const double* ga = Gs + 16 + i0 + perm - kq;  // A value of chunk c: ga[-4c]
            const double* wb = W + kq * 16;               // B value of chunk c: wb[64 c]
            doublex4_t acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
            double av[4], bv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                av[e] = ga[-4 * e];
                bv[e] = wb[64 * e];
            }
#pragma unroll 1
            for (int c = 0; c < nc; c += 4) {
                // operands of the next four chunks are read while these multiply (the last round
                // rereads its own)
                const int cn = c + 4 < nc ? c + 4 : c;
                double an[4], bn[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    an[e] = ga[-4 * (cn + e)];
                    bn[e] = wb[64 * (cn + e)];
                }
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[e], bv[e], acc0, 0, 0, 0);
                    acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[e + 1], bv[e + 1], acc1, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    av[e] = an[e];
                    bv[e] = bn[e];
                }
            }
            // ---- 3. steps 4q .. 4q + 3 of path p: x, and W1, Wperp and P of the step after each
            double z[4], x[4], w[4], pj[4], v[4];
            if (A.cache_perp) {
                const double* vp = Vs + (size_t(sub) * tlen + 4 * q) * 16 + m;
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = vp[16 * r];
            } else {
                path64_gauss<SRC>(A, lg, p, 1, q, z);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = fma(b, z[r], acc0[r] + acc1[r]);
                if constexpr (SRC == P64_CALLER) x[r] = path64_caller_x(x[r], 4 * q + r < N - 1);
                w[r] = W[(4 * q + 1 + r) * 16];
                pj[r] = P[4 * q + r];
            }
            if constexpr (MC) {
                path64_gauss<SRC>(A, lg, p, 2, q, z);
                const double nx = __shfl(z[0], lane + 16, 64);
                const double last = W20[(size_t(sub) * (tlen / 16 + 1) + rb + 1) * 16 + m];
                v[0] = z[1];
                v[1] = z[2];
                v[2] = z[3];
                v[3] = kq < 3 ? nx : last;
            }
#pragma unroll
            for (int g = 0; g < GREG; ++g) {
                if (g < job.gn) {
                    const double c1 = G[g].c1, al = G[g].al;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const double ap = al * pj[r];
                        const double e = exp2_32(e2, fma(c1, x[r], -ap));
                        f[g][0] = fma(e, e, f[g][0]);
                        f[g][1] = fma(e, w[r], f[g][1]);
                        if constexpr (MC) f[g][2] = fma(e, v[r], f[g][2]);
                        if constexpr (SIGNS == 2) {
                            const double d = exp2_32(e2, fma(-c1, x[r], -ap));
                            f[g][2] = fma(d, d, f[g][2]);
                            f[g][3] = fma(d, w[r], f[g][3]);
                        }
                    }
                }
                // one group's four chains at a time: interleaved groups cost 15 registers each
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- 4. sums over the path's lanes, then over the sub-tile's waves
#pragma unroll
        for (int g = 0; g < GREG; ++g)
            if (g < job.gn)
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const double t = sum_kq(f[g][s]);
                    if (kq == 0) red[((wave * GREG + g) * NS + s) * 16 + m] = t;
                }
        __syncthreads();
        for (int t = tid; t < job.gn << psh; t += NT) {
            const int g = t >> psh, pp = t & ((1 << psh) - 1);
            const int sb = pp >> 4, mm = pp & 15;
            if (pb + pp >= A.np) continue;
            const Path64Group Gr = G[g];
            double s[NS];
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                s[k] = 0.0;
                for (int u = 0; u < KW; ++u) s[k] += red[(((sb * KW + u) * GREG + g) * NS + k) * 16 + mm];
            }
            // step 0: v_0 = xi
            const double w0 = Ws[size_t(sb) * (tlen + 1) * 16 + mm];
            double* out = A.ints + (long(Gr.out) * A.np + pb + pp) * 2;
            const double Iv = Gr.dt * (Gr.xi * (1.0 + s[0]));
            const double Is = Gr.sdt * (Gr.sxi * (w0 + s[1]));
            if constexpr (MC) {
                const double Ip = Gr.sdt * (Gr.sxi * (W20[size_t(sb) * (tlen / 16 + 1) * 16 + mm] + s[2]));
                out[0] = Gr.rho * Is + Gr.crho * Ip - 0.5 * Iv;
                out[1] = 0.0;
            } else {
                out[0] = Iv;
                out[1] = Is;
                if constexpr (SIGNS == 2) {
                    double* o2 = A.ints2 + (long(Gr.out) * A.np + pb + pp) * 2;
                    o2[0] = Gr.dt * (Gr.xi * (1.0 + s[2]));
                    o2[1] = -(Gr.sdt * (Gr.sxi * (w0 + s[3])));
                }
            }
        }
        // the next job's first barrier comes before it writes red, and no wave reads Gs any more
    }
}

hipError_t launch_path64(const Path64Args& a, hipStream_t st) {
    const size_t lds = path64_lds_bytes(a);
    const int per = 16 * path64_subtiles(a.N);
    if (a.np < 1 || a.njobs < 1 || a.nsplit < 1 || a.N > PATH64_MFMA_MAX_N || a.np > path64_max_paths(a.N) || a.tlen != (a.N + 15) / 16 * 16)
        return hipErrorInvalidValue;
    const dim3 grid(unsigned((a.np + per - 1) / per), unsigned(a.nsplit));
    auto go = [&](auto kern) -> hipError_t {
        if (lds > 65536) {
            const hipError_t e = allow_lds(reinterpret_cast<const void*>(kern), lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, grid, dim3(unsigned(a.threads)), lds, st, a);
        return hipGetLastError();
    };
    auto pick = [&](auto greg, auto threads) -> hipError_t {
        constexpr int GREG = decltype(greg)::value, NT = decltype(threads)::value;
        auto from = [&](auto src) {
            constexpr int SRC = decltype(src)::value;
            return a.mc ? go(&k_path64<SRC, true, 1, GREG, NT>) : go(&k_path64<SRC, false, 1, GREG, NT>);
        };
        switch (a.src) {
            case P64_PHILOX: return from(std::integral_constant<int, P64_PHILOX>());
            case P64_MEMORY: return from(std::integral_constant<int, P64_MEMORY>());
            case P64_CALLER: return from(std::integral_constant<int, P64_CALLER>());
            default: return hipErrorInvalidValue;
        }
    };
    auto sized = [&](auto threads) -> hipError_t {
        if (a.signs == 2) {
            if (a.src != P64_PHILOX || a.mc || a.greg != 2) return hipErrorInvalidValue;
            return go(&k_path64<P64_PHILOX, false, 2, 2, decltype(threads)::value>);
        }
        if (a.greg == 2) return pick(std::integral_constant<int, 2>(), threads);
        if (a.greg == 4) return pick(std::integral_constant<int, 4>(), threads);
        if (a.greg == 8) return pick(std::integral_constant<int, 8>(), threads);
        return hipErrorInvalidValue;
    };
    if (a.threads == 512 && per == 16) return sized(std::integral_constant<int, 512>());
    return a.threads == 256 ? sized(std::integral_constant<int, 256>()) : hipErrorInvalidValue;
}

}  // namespace rb
