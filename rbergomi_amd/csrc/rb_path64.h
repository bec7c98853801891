// rb_path64.h -- tables and launchers of the single-pass FP64 path kernels (rb_path64.hip,
// rb_path64_fft.hip) and the FP64 payoff kernel (rb_payoff64.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rb_device.h"
#include "rb_types.h"

namespace rb {

// One distinct (H, eta, T, xi[, rho]) of a launch, ordered by unit: with x = Gamma*W1 + a W1 + b W1perp
// at step i and P the unit's row table, sqrt(v_{i+1} / xi) = 2^((c1 x - al P) / 32)
struct Path64Group {
    double c1;    // 16 log2(e) eta T^H sc
    double al;    // 16 log2(e) (eta^2 / 2) dt^2H, within [AL_MIN, AL_MAX]
    double xi, sxi;
    double dt, sdt;
    double rho, crho;  // plain MC only
    int out;           // the group's index in the integrals' array
    int pad;
};

// A unit (distinct H) and up to greg of its groups: one convolution of a path tile, and the
// integrals of these groups
struct Path64Job {
    int unit, g0, gn, pad;
};

// Row table entries past the last step, which make every group's integrand exactly zero there
// (al P = 1e10 / 32 octaves), and the bounds of al that keep al P finite there and without effect
// on the steps before (P <= 8192^2)
constexpr double P64_PAD = 1e40, P64_AL_MIN = 1e-30, P64_AL_MAX = 1e250;

// P64_MEMORY: Gaussians a kernel of the package left in Z (Sobol' points); P64_CALLER: a caller's
enum Path64Source { P64_PHILOX = 0, P64_MEMORY = 1, P64_CALLER = 2 };

// A caller's Gaussians may be anything.  What infinities and NaN do stays with their path and their steps, as
// it does in the direct sum: W1perp of the last step, which the model does not use, has no effect
// (`used`: the step has a successor), and an infinite exponent gives 0 or infinity, where exp2_32 would make NaN of it.
// The guards are compiled for P64_CALLER only: they cost the transform kernel 5 to 27% of its time (N = 256, M =
// 31250: 58 -> 68 us), which a caller's call, most of it the copy of its Gaussians, does not notice.
__host__ __device__ __forceinline__ double path64_caller_x(double x, bool used) {
    constexpr double BIG = 1e200;
    x = x > BIG ? BIG : x < -BIG ? -BIG : x;  // NaN stays
    return used ? x : 0.0;
}
// W1 beyond this (no Gaussian is) is not put through a transform, which would spread it over its path's other
// steps and the pair's other path
constexpr double P64_WILD = 64.0;

struct Path64Args {
    PhiloxKey key;
    long p0;               // Philox counter of the launch's path 0
    long np;               // paths
    int N;
    int njobs, nsplit;     // jobs, and the workgroups of a tile that share them
    int threads;           // per workgroup: 256 or 512
    int src;               // Path64Source
    int greg;              // groups per job at most (path64_greg)
    int mc, signs;         // plain MC; 2: the mirrored path's integrals too (ints2)
    int cache_perp;        // W1perp of the tile kept in LDS for the jobs after the first
    const double* Z;       // P64_MEMORY, P64_CALLER: path p at Z + p zstride, blocks of N values
    long zstride;
    const Unit* units;
    const double* gamma;   // [units][tlen]: a, Gamma_1 .. Gamma_{N-1}, 0 ..
    const double* ptab;    // [units][tlen]: P_{i+1} at i, P64_PAD from i = N - 1 on
    int tlen;              // N rounded up to 16
    const Path64Group* groups;
    const Path64Job* jobs;
    double* ints;          // [groups][np][2]: (integral of v, of sqrt(v) dW), plain MC (ln S_T, 0)
    double* ints2;
    // FFT kernel only
    const double2* tw;     // twiddles of both transforms (Fft64)
    const double2* ghat;   // [units][L] spectrum of gamma over L, in the middle pass's order
};

// gamma and ptab of every unit (off: 1 for the reference compensator ((i-1) dt)^2H, 0 for (i dt)^2H)
hipError_t launch_path64_tables(const Unit* units, int nunits, int N, int tlen, double off, double* gamma,
                                double* ptab, hipStream_t st);

// The matrix-core kernel (up to where path64_uses_fft may choose it): groups per job, launch shape, LDS
constexpr int PATH64_MFMA_MAX_N = 384;
int path64_greg(int groups_of_largest_unit, int signs);
void path64_shape(Path64Args& a, int cus);
size_t path64_lds_bytes(const Path64Args& a);
hipError_t launch_path64(const Path64Args& a, hipStream_t st);
// Paths one launch takes: HIP has no grid of 2^32 threads or more a dimension, and the product kernel spends up to
// 512 threads on 16 paths, the transform kernel 32 on a path (N <= 512) to 256 (N > 2048).  Larger requests go
// in chunks.
long path64_max_paths(int N);

// The transform kernel (N <= 4096, and whether it is taken): length 2^log2 >= 2N, twiddle and spectrum tables (path64_fft_table
// and L entries per unit), LDS
constexpr int PATH64_FFT_MAX_N = 4096, PATH64_FFT_MIN_LOG2 = 9;
bool path64_uses_fft(int N, int units, int groups, bool mc);
int path64_fft_log2(int N);
void path64_fft_shape(Path64Args& a, int cus);
long path64_fft_max_paths(int N);
size_t path64_fft_table(int N);
hipError_t launch_path64_fft_tables(const double* gamma, int nunits, int N, int tlen, double2* tw, double2* ghat,
                                    hipStream_t st);
hipError_t launch_path64_fft(const Path64Args& a, hipStream_t st);

}  // namespace rb
