// rb_hostmem.h -- pinned host blocks and streams that outlive the plan that used them.
//
// A one-shot pricing call otherwise spends more time on them than on its kernels: creating and
// destroying a stream took 85 + 27 us, allocating pinned memory about as much, and each copy
// from or to pageable memory waits for a staging copy (4 to 15 us; a small mixed-precision call made
// 16 of them).  Both pools are bounded, safe for several threads, and hold only idle objects: a
// stream or block goes back after its user has waited for the work on it.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <algorithm>

namespace rb {

// A pinned, coherent host block of at least the bytes asked for, from the pool (blocks are powers of two from
// 64 KiB; up to 64 MiB of idle blocks are kept), returned to it with the object.
class Pinned {
  public:
    Pinned() = default;
    Pinned(const Pinned&) = delete;
    Pinned& operator=(const Pinned&) = delete;
    ~Pinned() { release(); }
    // null if the memory cannot be had; the contents are undefined after it
    unsigned char* reserve(size_t bytes);
    void release();
    unsigned char* data() const { return p_; }

  private:
    unsigned char* p_ = nullptr;
    size_t bytes_ = 0;
};

// Tables of more bytes than this go to the device from the pageable memory they were made in, which the
// caller waits for: pinned memory is held for a plan's life and rounded up to a power of two (the exact sampler's
// factors are 134 MB for every H at N = 2048).
constexpr size_t PINNED_TABLES = size_t(4) << 20;

// n results a kernel wrote, in a pinned block or, where none could be had, in device memory; the caller has
// waited for the kernel
inline hipError_t fetch_results(double* to, const double* from, size_t n, bool pinned) {
    if (!to || n == 0) return hipSuccess;
    if (!pinned) return hipMemcpy(to, from, n * sizeof(double), hipMemcpyDeviceToHost);
    std::copy_n(from, n, to);
    return hipSuccess;
}

// A non-blocking stream of the current device; up to 32 idle ones are kept
hipError_t stream_get(hipStream_t* st);
// back to the pool of `device`: the stream is idle and not capturing
void stream_put(hipStream_t st, int device);

}  // namespace rb
