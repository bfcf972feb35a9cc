// Host memory in the place of a GPU: the entry points of the HIP runtime that
// the library's host code calls, for programs that check that code on a CPU.
// The .hip sources are compiled for the host only and linked with this file
// instead of the runtime.  Allocations are ordinary memory whose ranges are
// kept, copies run at once and check their ranges, kernels do not run: a launch
// calls on_launch with the kernel's mangled name and its arguments.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace hh {

// what a program sets
inline bool no_pinned = false;            // hipHostMalloc fails
inline long malloc_until = -1;            // hipMalloc fails once this many have succeeded (-1: never)
inline std::function<void(const char *, void **)> on_launch;
inline std::function<void(hipEvent_t)> on_event_wait;
inline std::function<float()> elapsed_ms; // between any two events
// what it reads
struct Copy {
    const void *dst, *src;
    size_t bytes;
};
inline std::vector<Copy> copies;          // hipMemcpyAsync calls

struct Range {
    size_t bytes;
    bool pinned;
};
inline std::map<const char *, Range> ranges;
inline std::map<const void *, std::string> names;
inline std::mutex mu;

inline void *allocate(size_t bytes, bool pinned) {
    char *const p = static_cast<char *>(calloc(bytes ? bytes : 1, 1));
    std::lock_guard<std::mutex> lock(mu);
    ranges[p] = Range{bytes, pinned};
    return p;
}
inline void release(void *p) {
    if (!p) return;
    std::lock_guard<std::mutex> lock(mu);
    if (!ranges.erase(static_cast<const char *>(p))) {
        printf("freed what was not allocated\n");
        abort();
    }
    free(p);
}
// The allocation that holds [p, p + bytes), or null.
inline const Range *range_of(const void *p, size_t bytes) {
    const char *const c = static_cast<const char *>(p);
    auto it = ranges.upper_bound(c);
    if (it == ranges.begin()) return nullptr;
    --it;
    return c + bytes <= it->first + it->second.bytes ? &it->second : nullptr;
}
inline bool on_device(const void *p, size_t bytes = 1) {
    std::lock_guard<std::mutex> lock(mu);
    const Range *const r = p ? range_of(p, bytes) : nullptr;
    return r && !r->pinned;
}
inline hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    if (!dst || !src) return hipErrorInvalidValue;
    if ((kind == hipMemcpyDeviceToHost && !on_device(src, bytes)) || (kind == hipMemcpyHostToDevice && !on_device(dst, bytes)) ||
        (kind == hipMemcpyDeviceToDevice && !(on_device(src, bytes) && on_device(dst, bytes)))) {
        printf("copy of %zu bytes outside an allocation\n", bytes);
        abort();
    }
    memcpy(dst, src, bytes);
    return hipSuccess;
}

#define HH_CHECK(x)                                                   \
    do {                                                              \
        if (!(x)) {                                                   \
            printf("%s:%d: %s is false\n", __FILE__, __LINE__, #x);   \
            return 1;                                                 \
        }                                                             \
    } while (0)

}  // namespace hh

extern "C" {

// kernel registration and launch (what the host side of a <<<>>> calls)
char __hip_fatbin[1];
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    hh::names[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static thread_local struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
} hh_call;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    hh_call = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = hh_call.grid;
    *block = hh_call.block;
    *lds = hh_call.lds;
    *s = hh_call.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **args, size_t, hipStream_t) {
    if (hh::on_launch) hh::on_launch(hh::names[fn].c_str(), args);
    return hipSuccess;
}

hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }

hipError_t hipMalloc(void **p, size_t n) {
    if (hh::malloc_until == 0) return hipErrorOutOfMemory;
    if (hh::malloc_until > 0) --hh::malloc_until;
    *p = hh::allocate(n, false);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    hh::release(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (hh::no_pinned) return hipErrorOutOfMemory;
    *p = hh::allocate(n, true);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    hh::release(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    memset(a, 0, sizeof *a);
    std::lock_guard<std::mutex> lock(hh::mu);
    const hh::Range *const r = hh::range_of(p, 1);
    a->type = r ? (r->pinned ? hipMemoryTypeHost : hipMemoryTypeDevice) : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind k) { return hh::copy(dst, src, n, k); }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind k, hipStream_t) {
    {
        std::lock_guard<std::mutex> lock(hh::mu);
        hh::copies.push_back({dst, src, n});
    }
    return hh::copy(dst, src, n, k);
}
hipError_t hipMemset(void *p, int v, size_t n) {
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (hh::on_event_wait) hh::on_event_wait(e);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = hh::elapsed_ms ? hh::elapsed_ms() : 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorInvalidValue; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorInvalidValue; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorInvalidValue; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorInvalidValue; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
