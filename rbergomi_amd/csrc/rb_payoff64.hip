// rb_payoff64.hip -- payoffs of a path's integrals and their block partial sums in FP64 (BS_call_price /
// posPart, rBergLib/rBergomiMT.cpp:383-391, 264-266), and the mixed-precision payoffs of the long-path
// kernel's integrals.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rb_fused.h"
#include "rb_math64.h"
#include "rb_payoff64.h"

namespace rb {

// the sum over a row of 16 lanes, in every lane of the row
__device__ __forceinline__ double row16_sum(double v) {
#define RB_ROR_ADD(n)                                                                              \
    {                                                                                              \
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + n, 0xf, 0xf, false); \
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + n, 0xf, 0xf, false); \
        v += __hiloint2double(hi, lo);                                                             \
    }
    RB_ROR_ADD(8)
    RB_ROR_ADD(4)
    RB_ROR_ADD(2)
    RB_ROR_ADD(1)
#undef RB_ROR_ADD
    return v;
}

// What a path's options share, and one payoff.  ints: NS values per (group, path).
struct PayRt64 {  // FP64 Romano-Touzi (Iv, Is)
    static constexpr int NS = 2;
    static constexpr bool TAB = true;
    PathRt64 q;
    __device__ __forceinline__ void set(const double* v, double rho) {
        q = path_rt64(v[0], v[1], rho);
    }
    __device__ __forceinline__ double pay(const double* e2, const PayOpt64& o) const { return rt_payoff64(e2, q, o.K, o.lnK); }
};
struct PayMc64 {  // FP64 plain MC (ln S_T, 0)
    static constexpr int NS = 2;
    static constexpr bool TAB = false;
    double S;
    __device__ __forceinline__ void set(const double* v, double) { S = exp(v[0]); }
    __device__ __forceinline__ double pay(const double*, const PayOpt64& o) const { return S - o.K > 0.0 ? S - o.K : 0.0; }
};
struct PayRtMix {  // mixed-precision Romano-Touzi (Iv, Is)
    static constexpr int NS = 2;
    static constexpr bool TAB = false;
    PathPG q;
    __device__ __forceinline__ void set(const double* v, double rho) {
        q.sig = sqrt((1.0 - rho * rho) * v[0]);
        q.lnS = -0.5 * rho * rho * v[0] + rho * v[1];
        pathpg_f32(q);
    }
    __device__ __forceinline__ double pay(const double*, const PayOpt64& o) const {
        return payoff_mixed(q, opt_f32(o.lnK, o.K), o.lnK);
    }
};
struct PayMcMix {  // plain MC (Iv, Is, Ip): ln S_T = rho Is + sqrt(1 - rho^2) Ip - Iv / 2
    static constexpr int NS = 3;
    static constexpr bool TAB = false;
    double S;
    __device__ __forceinline__ void set(const double* v, double rho) {
        S = exp(rho * v[1] + sqrt(1.0 - rho * rho) * v[2] - 0.5 * v[0]);
    }
    __device__ __forceinline__ double pay(const double*, const PayOpt64& o) const { return S - o.K > 0.0 ? S - o.K : 0.0; }
};

// Grid (blocks of 256 PPT paths, jobs).  A job is a run of options of one (group, rho): the fields
// they share (S', sigma, its reciprocal) are formed once per path, and an evaluation is the Mills
// pair and one exponential.  Vector-issue bound (about 75 FP64 instructions an evaluation, against
// some 280 with two library erfc, an exp and a square root each); PPT paths per thread share an
// option's row sums.  205 options on 2^19 paths: 0.91 -> 0.40 ms.  partial[(out*nblk_total + blk0 + blockIdx.x)*2] =
// (sum of payoffs, of squares); if payoff != nullptr the per-path payoffs are also written at
// payoff[p*out_size + out] (quadrature layout).
template <class Pay, int PPT>
__global__ void __launch_bounds__(256)
k_payoff64(const double* __restrict__ ints, long np, const PayJob64* __restrict__ jobs,
           const PayOpt64* __restrict__ opts, int out_size, long blk0, long nblk_total,
           double* __restrict__ partial, double* __restrict__ payoff) {
    __shared__ double e2[Pay::TAB ? EXP2_N : 1];
    __shared__ double sums[PAY64_OPTS][16][2];
    const int tid = threadIdx.x;
    if constexpr (Pay::TAB) load_exp2_tab(e2, tid, 256);
    const PayJob64 J = jobs[blockIdx.y];
    const long pb = long(blockIdx.x) * 256 * PPT + tid;
    Pay q[PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        const long p = pb + 256 * j;
        double v[3] = {0.01, 0.0, 0.0};
        if (p < np)
#pragma unroll
            for (int k = 0; k < Pay::NS; ++k) v[k] = ints[(long(J.group) * np + p) * Pay::NS + k];
        q[j].set(v, J.rho);
    }
    __syncthreads();
    for (int o = 0; o < J.n; ++o) {
        const PayOpt64 O = opts[J.o0 + o];
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            const long p = pb + 256 * j;
            double x = q[j].pay(e2, O);
            if (p >= np) x = 0.0;
            else if (payoff) payoff[p * out_size + O.out] = x;
            s1 += x;
            s2 = fma(x, x, s2);
        }
        s1 = row16_sum(s1);
        s2 = row16_sum(s2);
        if ((tid & 15) == 0) {
            sums[o][tid >> 4][0] = s1;
            sums[o][tid >> 4][1] = s2;
        }
    }
    __syncthreads();
    if (tid < 2 * J.n && partial) {
        const int o = tid >> 1, k = tid & 1;
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < 16; ++r) s += sums[o][r][k];
        partial[(long(opts[J.o0 + o].out) * nblk_total + blk0 + blockIdx.x) * 2 + k] = s;
    }
}

hipError_t launch_payoff64(const double* ints, long np, int ppt, const PayJob64* jobs, int njobs, const PayOpt64* opts,
                           int out_size, int kind, long blk0, long nblk_total, double* partial, double* payoff,
                           hipStream_t st) {
    const long per = 256L * ppt;
    const dim3 grid(unsigned((np + per - 1) / per), unsigned(njobs));
    auto go = [&](auto pay) -> hipError_t {
        using Pay = decltype(pay);
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, ints, np, jobs, opts, out_size, blk0, nblk_total, partial,
                               payoff);
            return hipGetLastError();
        };
        switch (ppt) {
            case 1: return launch(&k_payoff64<Pay, 1>);
            case 2: return launch(&k_payoff64<Pay, 2>);
            case 4: return launch(&k_payoff64<Pay, 4>);
            default: return hipErrorInvalidValue;
        }
    };
    switch (kind) {
        case PAY_RT64: return go(PayRt64());
        case PAY_MC64: return go(PayMc64());
        case PAY_RT_MIX: return go(PayRtMix());
        case PAY_MC_MIX: return go(PayMcMix());
        default: return hipErrorInvalidValue;
    }
}

}  // namespace rb
