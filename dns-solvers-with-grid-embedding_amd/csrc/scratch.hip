// scratch.hip -- working memory kept between the calls that write results out, and
// their copies to the host.
#include "scratch.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

using namespace dnsg;

namespace {

struct ScratchBlock {
    void *p;
    size_t bytes;
    int dev;
    bool used;
};
constexpr int BLOCKS = 64;
// blocks taken out of the pool under its lock, freed after it is released (declared before
// the lock): hipFree waits for the device, and other handles must not wait with it
struct Victims {
    void *p[BLOCKS];
    int n = 0;
    ~Victims();
};
struct ScratchPool {
    std::mutex m;
    std::condition_variable freed;
    ScratchBlock b[BLOCKS];
    int n = 0, users = 0;  // b[0, n): handed out or kept, the longest kept first
    int leaving = 0;       // victims not freed yet
    void drop(int i, Victims &v) {
        v.p[v.n++] = b[i].p;
        leaving++;
        std::move(b + i + 1, b + n, b + i);
        n--;
    }
    void trim(Victims &v) {
        for (int i = n - 1; i >= 0; i--)
            if (!b[i].used) drop(i, v);
    }
};
// never destroyed: handles may outlive the static objects of this library
ScratchPool &pool() {
    alignas(ScratchPool) static unsigned char room[sizeof(ScratchPool)];
    static ScratchPool &p = *new (room) ScratchPool;
    return p;
}
Victims::~Victims() {
    if (n == 0) return;
    for (int i = 0; i < n; i++) (void)hipFree(p[i]);
    std::lock_guard<std::mutex> l(pool().m);
    pool().leaving -= n;
    pool().freed.notify_all();
}

}  // namespace

// what other threads are freeing is waited for: their blocks are as good as kept ones to a
// caller that found no memory
void dnsg::scratch_trim() {
    {
        Victims v;
        std::lock_guard<std::mutex> l(pool().m);
        pool().trim(v);
    }
    std::unique_lock<std::mutex> l(pool().m);
    pool().freed.wait(l, [] { return pool().leaving == 0; });
}

void dnsg::scratch_users(int change) {
    Victims v;
    std::lock_guard<std::mutex> l(pool().m);
    pool().users += change;
    if (pool().users == 0) pool().trim(v);
}

hipError_t dnsg::scratch_available(size_t *bytes) {
    int dev = 0;
    size_t total = 0;
    ScratchPool &P = pool();
    std::unique_lock<std::mutex> l(P.m);  // held over the query: no block changes sides meanwhile
    P.freed.wait(l, [&] { return P.leaving == 0; });
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipMemGetInfo(bytes, &total);
    if (e != hipSuccess) return e;
    for (int i = 0; i < P.n; i++)
        if (!P.b[i].used && P.b[i].dev == dev) *bytes += P.b[i].bytes;
    return hipSuccess;
}

hipError_t dnsg::scratch_get(void **p, size_t bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    ScratchPool &P = pool();
    {
        // the smallest kept block that is large enough and no more than twice the size
        std::lock_guard<std::mutex> l(P.m);
        ScratchBlock *best = nullptr;
        for (int i = 0; i < P.n; i++) {
            ScratchBlock &c = P.b[i];
            if (!c.used && c.dev == dev && c.bytes >= bytes && c.bytes / 2 <= bytes && (!best || c.bytes < best->bytes)) best = &c;
        }
        if (best) {
            best->used = true;
            *p = best->p;
            return hipSuccess;
        }
    }
    e = dev_malloc(p, bytes);
    if (e != hipSuccess) return e;
    Victims v;
    std::lock_guard<std::mutex> l(P.m);
    if (P.n == BLOCKS)
        for (int i = 0; i < P.n; i++)
            if (!P.b[i].used) {
                P.drop(i, v);
                break;
            }
    if (P.n < BLOCKS) P.b[P.n++] = {*p, bytes, dev, true};  // else it is freed when given back
    return hipSuccess;
}

namespace {

void put_back(void *p) {
    ScratchPool &P = pool();
    Victims v;
    std::lock_guard<std::mutex> l(P.m);
    int i = 0;
    while (i < P.n && P.b[i].p != p) i++;
    if (i == P.n) {
        v.p[v.n++] = p;
        P.leaving++;
        return;
    }
    std::rotate(P.b + i, P.b + i + 1, P.b + P.n);
    ScratchBlock &mine = P.b[P.n - 1];
    mine.used = false;
    const int dev = mine.dev;
    size_t total = 0, kept = 0;
    if (hipDeviceTotalMem(&total, dev) != hipSuccess) total = 0;
    if (mine.bytes > total / 64) {  // never kept: the others stay
        P.drop(P.n - 1, v);
        return;
    }
    for (int j = 0; j < P.n; j++)
        if (!P.b[j].used && P.b[j].dev == dev) kept += P.b[j].bytes;
    for (int j = 0; j < P.n && kept > total / 64;) {  // the longest kept go first
        if (P.b[j].used || P.b[j].dev != dev) {
            j++;
            continue;
        }
        kept -= P.b[j].bytes;
        P.drop(j, v);
    }
}

}  // namespace

hipError_t dnsg::scratch_put(hipStream_t s, std::initializer_list<void *> ps) {
    const hipError_t e = hipStreamSynchronize(s);
    for (void *p : ps)
        if (p) put_back(p);
    return e;
}

// A plain copy into pageable memory runs at the rate of one host thread that also takes
// the page faults of a fresh array (4 to 10 GB/s against 57 of the link).  From two
// pieces on, the data comes through two pinned buffers instead: while the link fills one,
// a few threads move the other on (20 to 29 GB/s).  The buffers live for the call, about
// 0.5 ms, so a single piece (1.6 ms) is left to the plain copy; so is an array that the
// device can write itself (pinned or device memory).
hipError_t dnsg::copy_out(hipStream_t s, void *dst, const void *src, size_t bytes) {
    constexpr size_t PIECE = (size_t)16 << 20;
    hipPointerAttribute_t at;
    const bool pageable = hipPointerGetAttributes(&at, dst) != hipSuccess || at.type == hipMemoryTypeUnregistered;
    if (pageable) (void)hipGetLastError();  // an unknown pointer is an answer, not an error
    char *buf = nullptr;
    if (!pageable || bytes < 2 * PIECE || hipHostMalloc((void **)&buf, 2 * PIECE, hipHostMallocDefault) != hipSuccess) {
        if (pageable) (void)hipGetLastError();
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        const hipError_t w = hipStreamSynchronize(s);
        return e != hipSuccess ? e : w;
    }
    const int nt = (int)std::min(4u, std::max(1u, std::thread::hardware_concurrency()));
    const size_t pieces = (bytes + PIECE - 1) / PIECE;
    auto len = [&](size_t p) { return std::min(PIECE, bytes - p * PIECE); };
    auto fetch = [&](size_t p) {
        return hipMemcpyAsync(buf + (p & 1) * PIECE, static_cast<const char *>(src) + p * PIECE, len(p),
                              hipMemcpyDeviceToHost, s);
    };
    hipError_t e = fetch(0);
    for (size_t p = 0; p < pieces && e == hipSuccess; p++) {
        e = hipStreamSynchronize(s);
        if (e == hipSuccess && p + 1 < pieces) e = fetch(p + 1);
        if (e != hipSuccess) break;
        const size_t n = len(p);
        auto share = [&](int t) {
            const size_t a = n * t / nt, b = n * (t + 1) / nt;
            memcpy(static_cast<char *>(dst) + p * PIECE + a, buf + (p & 1) * PIECE + a, b - a);
        };
        std::thread th[4];
        for (int t = 1; t < nt; t++) {
            try {
                th[t] = std::thread(share, t);
            } catch (...) {  // no thread, or no memory for one, to be had
                share(t);
            }
        }
        share(0);
        for (int t = 1; t < nt; t++)
            if (th[t].joinable()) th[t].join();
    }
    const hipError_t w = hipStreamSynchronize(s);
    (void)hipHostFree(buf);
    return e != hipSuccess ? e : w;
}
