// Bookkeeping of csrc/scratch.hip on a host stand-in for the HIP runtime (hip_host/):
// scratch_test NAME runs one check and exits with 0 where it holds.
#include "../../dns-solvers-with-grid-embedding_amd/csrc/scratch.hip"

#include <cstdio>
#include <functional>
#include <string>

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #x); \
            exit(1);                                                 \
        }                                                            \
    } while (0)

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

int main(int argc, char **argv) {
    const std::map<std::string, std::function<void()>> tests = {
        {"waits_for_the_stream", waits_for_the_stream},
    };
    CHECK(argc == 2 && tests.count(argv[1]));
    scratch_users(1);
    tests.at(argv[1])();
    return 0;
}
