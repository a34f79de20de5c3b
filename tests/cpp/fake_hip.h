// A HIP runtime without a device for CPU checks of the host code: memory is a table of address
// ranges (never touched), every kernel launch succeeds and does nothing.  Include before
// blfid_host.cpp.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#define HIP_SYMBOL(x) (&(x))
#ifndef __align__
#define __align__(n) __attribute__((aligned(n)))
#endif

namespace fake {
struct Range {
    size_t bytes;
    unsigned long long id; // unique in the process, as the runtime's buffer ids
};
static std::map<size_t, Range> mem; // by address
static size_t limit = (size_t)64 << 30, used = 0;
static unsigned long long next_id = 1;
static long n_malloc = 0, n_free = 0, n_sync = 0;
static size_t copy_min = SIZE_MAX, copy_max = 0; // sizes of the synchronous copies
static hipError_t last = hipSuccess;

static hipError_t err(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
// the lowest gap that fits, so that freed addresses are handed out again
static hipError_t alloc(void **p, size_t bytes) {
    n_malloc++;
    const size_t sz = (bytes + 4095) & ~(size_t)4095;
    if (used + sz > limit) return err(hipErrorOutOfMemory);
    size_t at = (size_t)1 << 32;
    for (auto &kv : mem) {
        if (kv.first - at >= sz) break;
        at = kv.first + ((kv.second.bytes + 4095) & ~(size_t)4095);
    }
    mem[at] = {bytes, next_id++};
    used += sz;
    *p = (void *)at;
    return hipSuccess;
}
static hipError_t release(void *p) {
    n_free++;
    auto it = mem.find((size_t)p);
    if (it == mem.end()) return err(hipErrorInvalidValue);
    used -= (it->second.bytes + 4095) & ~(size_t)4095;
    mem.erase(it);
    return hipSuccess;
}
// hipDeviceReset: every allocation of the process is gone
static void reset() {
    mem.clear();
    used = 0;
}
} // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return fake::alloc(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return p ? fake::release(p) : hipSuccess; }
hipError_t hipMemcpy(void *d, const void *, size_t n, hipMemcpyKind k) {
    fake::copy_min = n < fake::copy_min ? n : fake::copy_min;
    fake::copy_max = n > fake::copy_max ? n : fake::copy_max;
    if (k == hipMemcpyDeviceToHost) std::memset(d, 0, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *, size_t n, hipMemcpyKind k, hipStream_t) {
    if (k == hipMemcpyDeviceToHost) std::memset(d, 0, n);
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = fake::limit - fake::used;
    *t = fake::limit;
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void *data, hipPointer_attribute a, hipDeviceptr_t p) {
    auto it = fake::mem.find((size_t)p);
    if (a != HIP_POINTER_ATTRIBUTE_BUFFER_ID || it == fake::mem.end()) return fake::err(hipErrorInvalidValue);
    *(unsigned *)data = (unsigned)it->second.id;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceSynchronize() { fake::n_sync++; return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = fake::last; fake::last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { *x = (hipGraphExec_t)1; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return hipSuccess; }
}
