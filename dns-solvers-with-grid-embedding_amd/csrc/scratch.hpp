// scratch.hpp -- device working memory of the output calls and copies to the host.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <initializer_list>

namespace dnsg {

// Working memory of the calls that write results out (budget, spectra, snapshots,
// checkpoints).  The driver clears a freed block before it hands it out again, so an
// allocation of the size just freed waits for that: 1 GB a call costs up to 30 ms where
// the kernels take 3.  Blocks given back are therefore kept for the next such call of
// any handle: at most 1/64 of the device's memory and 64 blocks, all freed with the last
// handle, and freed and tried again where an allocation finds no memory (dev_malloc).
// Safe with any number of threads.
hipError_t scratch_get(void **p, size_t bytes);
// gives blocks back (null ones are skipped) once stream s, the one that used them, has
// finished with them: the wait is made here, so that no path of a caller, an error's
// included, can leave a block to another handle while launches still use it; its status
hipError_t scratch_put(hipStream_t s, std::initializer_list<void *> ps);
void scratch_trim();
void scratch_users(int change);  // handles alive
// free memory of the current device, kept blocks included: dev_malloc finds them where
// nothing else is left, so whether and when they are freed does not change it
hipError_t scratch_available(size_t *bytes);
template <class T>
inline hipError_t scratch_get(T **p, size_t bytes) {
    return scratch_get(reinterpret_cast<void **>(p), bytes);
}
template <class T>
inline hipError_t dev_malloc(T **p, size_t bytes) {
    hipError_t e = hipMalloc(reinterpret_cast<void **>(p), bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        scratch_trim();
        e = hipMalloc(reinterpret_cast<void **>(p), bytes);
    }
    return e;
}
// device memory to the caller's array, in stream order; complete on return
hipError_t copy_out(hipStream_t s, void *dst, const void *src, size_t bytes);

}  // namespace dnsg
