// Bookkeeping of csrc/scratch.hip on a host stand-in for the HIP runtime (hip_host/):
// scratch_test NAME runs one check and exits with 0 where it holds.
#include "../../dns-solvers-with-grid-embedding_amd/csrc/scratch.hip"

#include <chrono>
#include <cstdio>
#include <functional>
#include <future>
#include <new>
#include <string>
#include <vector>

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #x); \
            exit(1);                                                 \
        }                                                            \
    } while (0)

// no host memory for a new thread, from the first wait for a piece on
static std::atomic<bool> no_memory{false};
void *operator new(size_t n) {
    void *p = no_memory ? nullptr : malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

static void *get(size_t bytes) {
    void *p = nullptr;
    CHECK(scratch_get(&p, bytes) == hipSuccess);
    return p;
}

// a block is handed on only after the stream that used it has finished
static void waits_for_the_stream() {
    ihipStream_t s;
    void *a = get(1000), *b = get(2000);
    s.busy = true;
    CHECK(scratch_put(&s, {nullptr, a, b}) == hipSuccess);
    CHECK(!s.busy);
    CHECK(get(1000) == a && get(2000) == b);  // kept
}

static ihipStream_t idle;
static void put(void *p) { CHECK(scratch_put(&idle, {p}) == hipSuccess); }
constexpr size_t MB = (size_t)1 << 20;  // a device of 1 GiB keeps 16

// a block that is too large to keep is freed alone
static void large_block_leaves_the_others() {
    void *a = get(4 * MB), *b = get(8 * MB), *c = get(20 * MB);
    put(a), put(b), put(c);
    CHECK(fake().in_use == 12 * MB);
    CHECK(get(4 * MB) == a && get(8 * MB) == b);
}

// over the limit, the blocks kept longest go, until the rest fits
static void oldest_go_first() {
    void *a = get(6 * MB), *b = get(7 * MB), *c = get(9 * MB);
    put(b), put(a), put(c);
    CHECK(fake().in_use == 15 * MB);
    CHECK(get(6 * MB) == a && get(9 * MB) == c);
}

// while a block is freed, other threads go on
static void try_another_thread() {
    fake().on_free = nullptr;
    std::promise<void> done;
    auto f = done.get_future();
    std::thread t([&] {
        void *p = nullptr;
        CHECK(scratch_get(&p, 100) == hipSuccess);
        done.set_value();
    });
    if (f.wait_for(std::chrono::seconds(5)) != std::future_status::ready) {
        printf("a second thread waits for the free\n");
        exit(1);
    }
    t.join();
}
static void frees_hold_no_lock() {
    void *a = get(20 * MB), *b = get(3 * MB);
    fake().on_free = try_another_thread;  // too large
    put(a);
    CHECK(!fake().on_free);
    put(b);
    fake().on_free = try_another_thread;  // on request
    scratch_trim();
    CHECK(!fake().on_free);
    put(get(10 * MB));
    put(get(5 * MB));
    fake().on_free = try_another_thread;  // over the limit
    put(get(12 * MB));
    CHECK(!fake().on_free);
    fake().on_free = try_another_thread;  // with the last handle
    scratch_users(-1);
    CHECK(!fake().on_free);
}

// an allocation that finds no memory waits for what another thread is freeing
static std::promise<void> freeing;
static void slow_free() {
    fake().on_free = nullptr;
    freeing.set_value();
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
}
static void allocation_waits_for_frees() {
    void *rest = nullptr, *p = nullptr;
    put(get(10 * MB));
    CHECK(hipMalloc(&rest, fake().total - 15 * MB) == hipSuccess);
    fake().on_free = slow_free;
    std::thread t(scratch_trim);
    freeing.get_future().wait();
    CHECK(dev_malloc(&p, 12 * MB) == hipSuccess);
    t.join();
}

// the calling thread moves what no other thread can be had for
static void copy_without_threads() {
    const size_t n = (size_t)37 << 20;
    std::vector<unsigned char> src(n), dst(n);
    for (size_t i = 0; i < n; i++) src[i] = (unsigned char)(i * 2654435761u >> 16);
    fake().on_sync = [] { no_memory = true; };
    const hipError_t e = copy_out(&idle, dst.data(), src.data(), n);
    no_memory = false;
    CHECK(e == hipSuccess && fake().host_buffers == 1 && dst == src);
}

// memory counts as available whether it is kept or free
static size_t available() {
    size_t n = 0;
    CHECK(scratch_available(&n) == hipSuccess);
    return n;
}
static void kept_memory_is_available() {
    const size_t all = fake().total;
    void *a = get(10 * MB);
    CHECK(available() == all - 10 * MB);
    put(a);
    CHECK(fake().in_use == 10 * MB && available() == all);
    CHECK(get(8 * MB) == a && available() == all - 10 * MB);
    put(a);
    // what an allocation takes, also where it empties the pool
    void *p = nullptr;
    CHECK(dev_malloc(&p, all - 4 * MB) == hipSuccess);
    CHECK(available() == 4 * MB);
    CHECK(hipFree(p) == hipSuccess && available() == all);
}

// which way a copy goes, and that it is whole: one plain copy below two pieces of 16 MiB;
// from there on through one pinned buffer, a copy a piece, the last of any length
static void copies_of_every_length() {
    const size_t piece = 16 * MB;
    const struct {
        size_t bytes, pieces;  // pieces 0: the plain copy
    } cases[] = {{1, 0}, {piece, 0}, {2 * piece - 1, 0}, {2 * piece, 2}, {2 * piece + 1, 3}, {2 * piece + 3, 3},
                 {3 * piece - 1, 3}, {3 * piece, 3}, {3 * piece + 7, 4}};
    for (const auto &c : cases) {
        std::vector<unsigned char> src(c.bytes), dst(c.bytes + 64, 0xa5);
        for (size_t i = 0; i < c.bytes; i++) src[i] = (unsigned char)(i * 2654435761u >> 16);
        fake().copies = fake().host_buffers = 0;
        CHECK(copy_out(&idle, dst.data(), src.data(), c.bytes) == hipSuccess);
        CHECK(fake().host_buffers == (c.pieces ? 1 : 0) && fake().copies == (c.pieces ? c.pieces : 1));
        CHECK(memcmp(dst.data(), src.data(), c.bytes) == 0);
        for (size_t i = 0; i < 64; i++) CHECK(dst[c.bytes + i] == 0xa5);
    }
}

int main(int argc, char **argv) {
    const std::map<std::string, std::function<void()>> tests = {
        {"waits_for_the_stream", waits_for_the_stream},
        {"large_block_leaves_the_others", large_block_leaves_the_others},
        {"oldest_go_first", oldest_go_first},
        {"frees_hold_no_lock", frees_hold_no_lock},
        {"allocation_waits_for_frees", allocation_waits_for_frees},
        {"copy_without_threads", copy_without_threads},
        {"copies_of_every_length", copies_of_every_length},
        {"kept_memory_is_available", kept_memory_is_available},
    };
    CHECK(argc == 2 && tests.count(argv[1]));
    no_memory = true;  // the first handle asks for none
    scratch_users(1);
    no_memory = false;
    tests.at(argv[1])();
    return 0;
}
