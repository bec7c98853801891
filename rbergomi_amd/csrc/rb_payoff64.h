// rb_payoff64.h -- work tables and launchers of the FP64 payoff stage (rb_payoff64.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

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

// FP64 payoffs of (Iv, Is) or (ln S_T, 0) per path; mixed-precision ones of (Iv, Is) or (Iv, Is, Ip)
enum PayKind { PAY_RT64, PAY_MC64, PAY_RT_MIX, PAY_MC_MIX };

// Paths per payoff thread, so that a block's sums cover 256 times as many paths: as many as leave
// 2048 blocks of the whole option table, at most 4
inline int payoff_paths_per_thread(long M, int nopt) {
    int ppt = 4;
    while (ppt > 1 && M / (256L * ppt) * ((nopt + PAY64_OPTS - 1) / PAY64_OPTS) < 2048) ppt /= 2;
    return ppt;
}

// Jobs of up to PAY64_OPTS options of one (group, rho), shorter where nblk path blocks alone leave
// some of the compute units without one; options in the order given, equal (group, rho) adjacent
struct PayRow {
    int group, out;
    double rho, K, lnK;
};
void payoff_jobs(const std::vector<PayRow>& rows, long nblk, int cus, std::vector<PayJob64>& jobs,
                 std::vector<PayOpt64>& opts);

// ppt: paths per thread (1, 2 or 4); a partial sum covers 256 ppt paths
hipError_t launch_payoff64(const double* ints, long np, int ppt, const PayJob64* jobs, int njobs, const PayOpt64* opts,
                           int out_size, int kind, long blk0, long nblk_total, double* partial, double* payoff,
                           hipStream_t st);

}  // namespace rb
