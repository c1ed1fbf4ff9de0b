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
int known_destination(char* dst, bool device) {
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
    (void)device;
    sfv::staging_release();
    return 0;
}
int device_destination() { return known_destination(stub::device_alloc(20 * MB), true); }
int pinned_destination() {
    void* p = nullptr;
    CHECK(hipHostMalloc(&p, 20 * MB, hipHostMallocDefault) == hipSuccess);
    return known_destination((char*)p, false);
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "pageable") return pageable();
    if (what == "device_destination") return device_destination();
    if (what == "pinned_destination") return pinned_destination();
    std::printf("unknown scenario\n");
    return 2;
}
