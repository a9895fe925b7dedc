// The few HIP runtime calls of csrc/scratch.hip on host memory, so that its bookkeeping (and
// plain host code of other headers) can be tested without a GPU.  A test sets the device's
// size and reads what was done.
#pragma once
#include <pthread.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <map>
#include <mutex>

#define __host__
#define __device__
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
struct ihipStream_t {
    std::atomic<bool> busy{false};  // launches in flight
};
typedef ihipStream_t *hipStream_t;
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
enum { hipHostMallocDefault = 0 };

struct FakeDevice {
    std::recursive_mutex m;
    size_t total = (size_t)1 << 30, in_use = 0;
    std::map<void *, size_t> blocks;
    void (*on_free)() = nullptr;  // called by hipFree
    void (*on_sync)() = nullptr;        // called by hipStreamSynchronize
    size_t copies = 0, host_buffers = 0;
};
inline FakeDevice &fake() {
    static FakeDevice d;
    return d;
}

inline hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipDeviceTotalMem(size_t *b, int) { return *b = fake().total, hipSuccess; }
inline hipError_t hipMemGetInfo(size_t *free, size_t *total) {
    std::lock_guard<std::recursive_mutex> l(fake().m);
    return *total = fake().total, *free = fake().total - fake().in_use, hipSuccess;
}
inline hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> l(fake().m);
    if (fake().in_use + bytes > fake().total) return hipErrorOutOfMemory;
    *p = malloc(64);  // an address; no test touches what it points to
    fake().blocks[*p] = bytes;
    fake().in_use += bytes;
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    if (fake().on_free) fake().on_free();
    std::lock_guard<std::recursive_mutex> l(fake().m);
    const auto it = fake().blocks.find(p);
    if (it == fake().blocks.end()) return hipErrorInvalidValue;
    fake().in_use -= it->second;
    fake().blocks.erase(it);
    free(p);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->busy = false;
    if (fake().on_sync) fake().on_sync();
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    fake().copies++;
    memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, int) {
    fake().host_buffers++;
    return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    return a->type = hipMemoryTypeUnregistered, hipSuccess;
}
