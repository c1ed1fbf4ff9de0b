// copy_to_host (sfv_transfer.hip) over the CPU stand-in for the HIP runtime;
// the scenario is the first argument.  Ends with 0 if it held.
#include <cstdio>
#include <string>
#include <vector>

#include "sfv_transfer.hip"

namespace {

constexpr size_t MB = (size_t)1 << 20;

#define CHECK(cond)                                                     \
    do {                                                                \
        if (!(cond)) {                                                  \
            std::printf("line %d: %s\n", __LINE__, #cond);              \
            return 1;                                                   \
        }                                                               \
    } while (0)

struct Source {
    size_t n;
    char* dev;
    std::vector<char> want;
    explicit Source(size_t bytes) : n(bytes), dev(stub::device_alloc(bytes)), want(bytes) {
        for (size_t k = 0; k < n; ++k) want[k] = (char)(k * 2654435761u >> 13);
    }
    // the bytes arrive by work still queued on st
    void queue_on(hipStream_t st) {
        st->pending = [this] { stub::with_access(dev, n, [&] { std::memcpy(dev, want.data(), n); }); };
    }
};

int bytes_of(size_t n) {
    Source s(n);
    StubStream st;
    s.queue_on(&st);
    std::vector<char> out(n + 2, 7);
    CHECK(sfv::copy_to_host(out.data() + 1, s.dev, n, &st) == hipSuccess);
    CHECK(std::memcmp(out.data() + 1, s.want.data(), n) == 0);
    CHECK(out[0] == 7 && out[n + 1] == 7);
    return 0;
}

int pageable() {
    sfv::staging_retain();
    for (size_t n : {(size_t)1, 8 * MB - 1, 8 * MB, 8 * MB + 1, 16 * MB, 16 * MB + 3, 33 * MB + 5})
        if (bytes_of(n)) return 1;
    sfv::staging_release();
    return 0;
}

// Memory the runtime knows is written by one copy of its own.
int known_destination(char* dst) {
    sfv::staging_retain();
    Source s(20 * MB);
    StubStream st;
    s.queue_on(&st);
    const long allocs = stub::host_allocs;
    CHECK(sfv::copy_to_host(dst, s.dev, s.n, &st) == hipSuccess);
    CHECK(stub::copies == 1 && st.copies == 1);
    CHECK(stub::host_allocs == allocs);
    int differs = 0;
    stub::with_access(dst, s.n, [&] { differs = std::memcmp(dst, s.want.data(), s.n); });
    CHECK(differs == 0);
    sfv::staging_release();
    return 0;
}
int device_destination() { return known_destination(stub::device_alloc(20 * MB)); }
int pinned_destination() {
    void* p = nullptr;
    CHECK(hipHostMalloc(&p, 20 * MB, hipHostMallocDefault) == hipSuccess);
    return known_destination((char*)p);
}

// The caller's stream only waits: the copies run on another.
int callers_stream() {
    sfv::staging_retain();
    Source s(20 * MB);
    StubStream st;
    s.queue_on(&st);
    std::vector<char> out(s.n);
    CHECK(sfv::copy_to_host(out.data(), s.dev, s.n, &st) == hipSuccess);
    CHECK(std::memcmp(out.data(), s.want.data(), s.n) == 0);
    CHECK(stub::copies >= 10);                    // staged
    CHECK(st.copies == 0 && st.events == 0);
    sfv::staging_release();
    return 0;
}

// Handles made, read and destroyed one after the other share one lane; the
// first that goes without having read as much gives it back.
int one_after_the_other() {
    for (int k = 0; k < 5; ++k) {
        sfv::staging_retain();
        CHECK(bytes_of(12 * MB) == 0);
        sfv::staging_release();
        CHECK(stub::host_allocs == 1 && stub::host_live == 1 && stub::streams_live == 1);
    }
    sfv::staging_retain();
    CHECK(bytes_of(MB) == 0);
    CHECK(stub::host_live == 1);
    sfv::staging_release();
    CHECK(stub::host_live == 0 && stub::streams_live == 0 && stub::events_live == 0);
    return 0;
}

// Threads that copy at once have at most MAX_LANES lanes; one is left at most.
int many_at_once() {
    constexpr int T = 9;
    for (int k = 0; k < T; ++k) sfv::staging_retain();
    std::atomic<int> bad{0};
    std::vector<std::thread> threads;
    for (int k = 0; k < T; ++k)
        threads.emplace_back([&] {
            for (int r = 0; r < 3; ++r) bad += bytes_of(17 * MB + 1);
        });
    for (auto& t : threads) t.join();
    CHECK(bad == 0);
    CHECK(stub::host_live <= 4 && stub::streams_live <= 4);
    for (int k = 0; k < T; ++k) sfv::staging_release();
    CHECK(stub::host_live <= 1 && stub::streams_live <= 1);
    return 0;
}

// A copy that fails ends with its error, with no thread left, and the next works.
int failing() {
    sfv::staging_retain();
    Source s(40 * MB);
    StubStream st;
    s.queue_on(&st);
    std::vector<char> out(s.n);
    for (long k : {0L, 3L, 8L, 19L}) {
        stub::fail_copy = k;
        CHECK(sfv::copy_to_host(out.data(), s.dev, s.n, &st) == hipErrorUnknown);
    }
    stub::fail_copy = -1;
    CHECK(sfv::copy_to_host(out.data(), s.dev, s.n, &st) == hipSuccess);
    CHECK(std::memcmp(out.data(), s.want.data(), s.n) == 0);
    sfv::staging_release();
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "pageable") return pageable();
    if (what == "device_destination") return device_destination();
    if (what == "pinned_destination") return pinned_destination();
    if (what == "callers_stream") return callers_stream();
    if (what == "one_after_the_other") return one_after_the_other();
    if (what == "many_at_once") return many_at_once();
    if (what == "failing") return failing();
    std::printf("unknown scenario\n");
    return 2;
}
