// rb_payoff64.h -- work tables and launchers of the FP64 payoff stage (rb_payoff64.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "rb_types.h"

namespace rb {

constexpr int PAY64_OPTS = 32;  // options per job at most

// options [o0, o0 + n) of the PayOpt64 table, all of one group and rho
struct PayJob64 {
    int group, o0, n, pad;
    double rho;
};
struct PayOpt64 {
    double K, lnK;
    int out, pad;
};

// ppt: paths per thread (1, 2 or 4); a partial sum covers 256 ppt paths
hipError_t launch_payoff64(const double* ints, long np, int ppt, const PayJob64* jobs, int njobs, const PayOpt64* opts,
                           int out_size, int method, long blk0, long nblk_total, double* partial, double* payoff,
                           hipStream_t st);

}  // namespace rb
