// rb_lanes.h -- threads of one path pair: their barrier and their sums (rb_path64_fft.hip,
// rb_fused_fft.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace rb {

struct BlockSync {
    __device__ __forceinline__ void operator()() const { __syncthreads(); }
};
// threads of one wave: LDS operations of a wave complete in order, so only the compiler is held
struct WaveSync {
    __device__ __forceinline__ void operator()() const {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// Sum v[0 .. V) over W lanes (V a power of two): each of log2 V steps hands half of the values to the
// partner lane, so that a lane ends with one value of index `idx`, summed over all W lanes.
template <int W, int V>
__device__ __forceinline__ double lanes_sum(double (&v)[V], int lane, int& idx) {
    int off = W / 2;
    idx = 0;
#pragma unroll
    for (int n = V / 2; n >= 1; n >>= 1, off >>= 1) {
        const bool hi = lane & off;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const double send = hi ? v[i] : v[i + n], keep = hi ? v[i + n] : v[i];
            v[i] = keep + __shfl_xor(send, off, 64);
        }
        idx = 2 * idx + (hi ? 1 : 0);
    }
    double s = v[0];
#pragma unroll
    for (; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

}  // namespace rb
