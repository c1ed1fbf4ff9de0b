// The part of the HIP runtime that sfv_transfer.hip uses, on the CPU: copies
// run at once, a stream's work pending before a copy (stub::pending) runs when
// the stream is next used or waited for, and what is called is counted.
// "Device" memory is mapped without access, so that touching it from the host
// ends the program.
#pragma once

#include <sys/mman.h>

#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipStreamNonBlocking = 1 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2, hipMemoryTypeManaged = 3 };
struct hipPointerAttribute_t {
    hipMemoryType type;
    int device;
    void *devicePointer, *hostPointer;
};
struct StubStream {
    std::function<void()> pending;
    std::atomic<long> copies{0}, events{0};
};
using hipStream_t = StubStream*;
using hipEvent_t = int*;

namespace stub {
inline std::mutex mu;
inline std::map<char*, std::pair<size_t, hipMemoryType>> known;   // what the runtime allocated
inline std::atomic<long> host_allocs{0}, host_live{0}, streams_live{0}, events_live{0}, copies{0};
inline std::atomic<long> fail_copy{-1};                           // the copy that fails, counted from now
inline std::pair<size_t, hipMemoryType> find(const void* p) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = known.upper_bound((char*)p);
    if (it == known.begin()) return {0, hipMemoryTypeUnregistered};
    --it;
    return (char*)p < it->first + it->second.first ? it->second : std::pair<size_t, hipMemoryType>{0, hipMemoryTypeUnregistered};
}
inline void drain(hipStream_t s) {
    if (s && s->pending) {
        auto f = std::move(s->pending);
        s->pending = nullptr;
        f();
    }
}
inline char* device_alloc(size_t n) {
    char* p = (char*)mmap(nullptr, n, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    std::lock_guard<std::mutex> lk(mu);
    known[p] = {n, hipMemoryTypeDevice};
    return p;
}
// let the "runtime" at device memory
template <class F>
void with_access(const void* p, size_t n, F&& f) {
    const bool dev = find(p).second == hipMemoryTypeDevice;
    if (dev) mprotect((void*)((size_t)p & ~(size_t)4095), n + ((size_t)p & 4095), PROT_READ | PROT_WRITE);
    f();
    if (dev) mprotect((void*)((size_t)p & ~(size_t)4095), n + ((size_t)p & 4095), PROT_NONE);
}
}  // namespace stub

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    *a = {stub::find(p).second, 0, nullptr, nullptr};
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    std::lock_guard<std::mutex> lk(stub::mu);
    stub::known[(char*)*p] = {n, hipMemoryTypeHost};
    ++stub::host_allocs;
    ++stub::host_live;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    {
        std::lock_guard<std::mutex> lk(stub::mu);
        stub::known.erase((char*)p);
    }
    std::free(p);
    --stub::host_live;
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = new StubStream;
    ++stub::streams_live;
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
    delete s;
    --stub::streams_live;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { stub::drain(s); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    stub::drain(s);
    ++s->copies;
    ++stub::copies;
    if (stub::fail_copy >= 0 && stub::fail_copy-- == 0) return hipErrorUnknown;
    stub::with_access(dst, n, [&] { stub::with_access(src, n, [&] { std::memcpy(dst, src, n); }); });
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new int(0); ++stub::events_live; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; --stub::events_live; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { stub::drain(s); ++s->events; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
