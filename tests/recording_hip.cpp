// A HIP runtime for the host half of the library on a machine without a GPU: memory is the host's,
// copies are memcpy, streams and events do nothing, and kernels are not run but recorded (name, grid,
// block, dynamic LDS), after the check the runtime itself makes of a launch (hip_runtime_api.h: every
// dimension's gridDim * blockDim below 2^32).  Loaded with global visibility before the library, whose
// calls then end here.
#include <hip/hip_runtime.h>

#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <mutex>
#include <string>

#include "rb_fused.h"
#include "rb_path64.h"

namespace {
std::mutex mu;
std::map<const void*, std::string> names;
std::map<void*, size_t> mapped;
std::string record;           // a line per launch
size_t pinned_now, pinned_most, pinned_fail = SIZE_MAX;
unsigned pinned_flags = ~0u;  // the flags every pinned block had
hipError_t last = hipSuccess;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t st;
} config;

hipError_t result(hipError_t e) { return last = e; }
// address space alone: pages come with the first write
void* get(size_t bytes) {
    void* p = mmap(nullptr, bytes ? bytes : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    mapped[p] = bytes ? bytes : 1;
    return p;
}
size_t put(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = mapped.find(p);
    if (it == mapped.end()) return 0;
    const size_t n = it->second;
    munmap(p, n);
    mapped.erase(it);
    return n;
}
}  // namespace

extern "C" {
// ---- what a test asks for
const char* rec_launches() { return record.c_str(); }
void rec_clear() { record.clear(); }
size_t rec_pinned_most() { return pinned_most; }
unsigned rec_pinned_flags() { return pinned_flags; }
void rec_fail_pinned_from(size_t bytes) { pinned_fail = bytes; }  // pinned blocks of so many bytes cannot be had

// ---- the runtime
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    p->sharedMemPerBlock = p->maxSharedMemoryPerMultiProcessor = 160 * 1024;
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error of the recording runtime"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) {
    *p = nullptr;
    return hipSuccess;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return result((*p = get(n)) ? hipSuccess : hipErrorOutOfMemory); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    static std::map<const void*, void*> at;
    void*& a = at[symbol];
    if (!a) a = get(size_t(1) << 30);
    *p = a;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    put(p);
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) { return hipFree(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (n >= pinned_fail) return result(hipErrorOutOfMemory);
    pinned_flags &= flags;
    pinned_now += n;
    if (pinned_now > pinned_most) pinned_most = pinned_now;
    return hipMalloc(p, n);
}
hipError_t hipHostFree(void* p) {
    pinned_now -= put(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.f;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

// ---- kernels
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    config = Config{grid, block, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *st = config.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, hipStream_t) {
    const auto over = [](unsigned n, unsigned m) { return n < 1 || m < 1 || uint64_t(n) * m >= uint64_t(1) << 32; };
    if (over(g.x, b.x) || over(g.y, b.y) || over(g.z, b.z) || uint64_t(b.x) * b.y * b.z > 1024 || lds > 160 * 1024)
        return result(hipErrorInvalidConfiguration);
    const std::string& name = names[f];
    record += name + " grid " + std::to_string(g.x) + " " + std::to_string(g.y) + " block " + std::to_string(b.x) +
              " lds " + std::to_string(lds);
    if (name.find("k_path64I") != std::string::npos || name.find("k_path64_fftI") != std::string::npos) {
        const rb::Path64Args& a = *static_cast<const rb::Path64Args*>(args[0]);
        record += " p0 " + std::to_string(a.p0) + " np " + std::to_string(a.np) + " njobs " + std::to_string(a.njobs) +
                  " nsplit " + std::to_string(a.nsplit) + " perp " + std::to_string(a.cache_perp) +
                  " mH0 " + std::to_string(int(1e6 * a.units[0].H + 0.5));
    }
    if (name.find("k_fusedI") != std::string::npos)
        record += " items " + std::to_string(static_cast<const rb::FusedBatchArgs*>(args[0])->total_items);
    // results to tell apart: price I + 1, standard error I + 1001, vol I + 2001
    if (name.find("k_reduce_iv") != std::string::npos)
        for (int k = 0; k < 3; ++k)
            for (unsigned I = 0; I < g.x; ++I)
                if (double* out = *static_cast<double**>(args[3 + k])) out[I] = 1000.0 * k + I + 1;
    record += "\n";
    return hipSuccess;
}
}
