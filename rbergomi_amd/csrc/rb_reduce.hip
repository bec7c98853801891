// rb_reduce.hip -- prices, standard errors and implied vols from partial sums (price = S/M,
// stat = sqrt(S2/M - price^2)/sqrt(M), rBergLib/rBergomiMT.cpp:404-409; IV_call, :421-423).
#include <hip/hip_runtime.h>

#include "rb_iv.h"
#include "rb_kernels.h"

namespace rb {

// One workgroup per output row: ordered strided sums of its (sum, sum of squares) pairs, then a fixed
// tree (deterministic), then the row's implied vol by the whole workgroup.  Latency-bound: with one
// thread solving each vol it took 36 us of a mixed-precision request of 21 rows (with its pricing
// kernel at 31), 34 us for 205 rows and 46 for 250; now 8.5 us for the 21.
__global__ void __launch_bounds__(256)
k_reduce_iv(const double* __restrict__ partial, ReduceRows rows, const Option* __restrict__ opts,
            double* __restrict__ price, double* __restrict__ stat, double* __restrict__ iv, int* __restrict__ counter) {
    __shared__ IvShared sh;
    const int I = blockIdx.x;
    const long n = rows.n ? rows.n[I] : rows.all_n;
    const double* base = partial + (rows.off ? rows.off[I] : 2 * n * I);
    double a = 0.0, b = 0.0;
    for (long k = threadIdx.x; k < n; k += 256) {
        a += base[2 * k];
        b += base[2 * k + 1];
    }
    block_sum_pair(a, b, sh);
    const double m = double(rows.M ? rows.M[I] : rows.all_M);
    const double pr = a / m;
    if (threadIdx.x == 0) {
        price[I] = pr;
        stat[I] = sqrt(b / m - pr * pr) / sqrt(m);
        if (counter && I == 0) *counter = 0;
    }
    if (!iv) return;
    const double v = implied_vol_block(pr, opts[I].K, opts[I].lnK, opts[I].T, sh);
    if (threadIdx.x == 0) iv[I] = v;
}

hipError_t launch_reduce_iv(const double* partial, const ReduceRows& rows, const Option* opts, int nrows, double* price,
                            double* stat, double* iv, int* counter, hipStream_t st) {
    if (nrows < 1) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_iv, dim3(unsigned(nrows)), dim3(256), 0, st, partial, rows, opts, price, stat, iv,
                       counter);
    return hipGetLastError();
}

// implied vols of prices that were adjusted after their reduction
__global__ void __launch_bounds__(256)
k_iv(const double* __restrict__ price, const Option* __restrict__ opts, double* __restrict__ iv) {
    __shared__ IvShared sh;
    const int I = blockIdx.x;
    const double v = implied_vol_block(price[I], opts[I].K, opts[I].lnK, opts[I].T, sh);
    if (threadIdx.x == 0) iv[I] = v;
}

hipError_t launch_iv(const double* price, const Option* opts, int nrows, double* iv, hipStream_t st) {
    hipLaunchKernelGGL(k_iv, dim3(unsigned(nrows)), dim3(256), 0, st, price, opts, iv);
    return hipGetLastError();
}

}  // namespace rb
