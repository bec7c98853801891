// rb_hostmem.cpp -- pools of pinned host blocks and streams (rb_hostmem.h).
#include "rb_hostmem.h"

#include <map>
#include <mutex>
#include <vector>

namespace rb {

namespace {
constexpr size_t PINNED_MIN = size_t(64) << 10, PINNED_KEEP = size_t(64) << 20;
constexpr size_t STREAMS_KEEP = 32;

// not destroyed at exit: the HIP runtime may be gone by then
struct Pools {
    std::mutex mu;
    std::multimap<size_t, unsigned char*> blocks;
    size_t block_bytes = 0;
    std::vector<std::pair<int, hipStream_t>> streams;
};
Pools& pools() {
    static Pools* p = new Pools();
    return *p;
}
}  // namespace

unsigned char* Pinned::reserve(size_t bytes) {
    if (p_ && bytes_ >= bytes) return p_;
    release();
    size_t want = PINNED_MIN;
    while (want < bytes) want *= 2;
    {
        Pools& P = pools();
        std::lock_guard<std::mutex> lock(P.mu);
        const auto it = P.blocks.find(want);
        if (it != P.blocks.end()) {
            p_ = it->second;
            bytes_ = want;
            P.blocks.erase(it);
            P.block_bytes -= want;
            return p_;
        }
    }
    void* p = nullptr;
    // coherent whatever HIP_HOST_COHERENT says: kernels write results here, and the host reads them after an event
    // or a stream alone
    if (hipHostMalloc(&p, want, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    p_ = static_cast<unsigned char*>(p);
    bytes_ = want;
    return p_;
}

void Pinned::release() {
    if (!p_) return;
    {
        Pools& P = pools();
        std::lock_guard<std::mutex> lock(P.mu);
        if (P.block_bytes + bytes_ <= PINNED_KEEP) {
            P.blocks.emplace(bytes_, p_);
            P.block_bytes += bytes_;
            p_ = nullptr;
            bytes_ = 0;
            return;
        }
    }
    (void)hipHostFree(p_);
    p_ = nullptr;
    bytes_ = 0;
}

hipError_t stream_get(hipStream_t* st) {
    int device = 0;
    const hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    {
        Pools& P = pools();
        std::lock_guard<std::mutex> lock(P.mu);
        for (auto it = P.streams.rbegin(); it != P.streams.rend(); ++it)
            if (it->first == device) {
                *st = it->second;
                P.streams.erase(std::next(it).base());
                return hipSuccess;
            }
    }
    return hipStreamCreateWithFlags(st, hipStreamNonBlocking);
}

void stream_put(hipStream_t st, int device) {
    {
        Pools& P = pools();
        std::lock_guard<std::mutex> lock(P.mu);
        if (P.streams.size() < STREAMS_KEEP) {
            P.streams.push_back({device, st});
            return;
        }
    }
    (void)hipStreamDestroy(st);
}

}  // namespace rb
