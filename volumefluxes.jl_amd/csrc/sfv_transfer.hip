// sfv_transfer.hip — device-to-host copies into pageable memory.
//
// hipMemcpy to pageable memory runs at 18 GB/s where the destination's pages
// are mapped and at 4 to 10 GB/s where they are fresh (a new array's pages are
// mapped one fault at a time), against 57 GB/s into pinned memory.  A copy
// here goes through a ring of pinned slots: the calling thread queues the DMA
// of the next chunks while worker threads empty the slots that have arrived,
// so the copies and page faults of several threads overlap with the DMA.
// Measured, us for the plain copy and this one: 9 MB mapped 535 and 330; 20 MB
// 1100 and 550; 35 MB 2000 and 920, fresh 3500 and 1350; 101 MB 5800 and 2550,
// fresh 9800 and 2900.
//
// The slots belong to a lane, one lane per copy under way, with a stream of its
// own; at most MAX_LANES lanes exist in the process (64 MB), made on first use.
// A copy that finds none free is a plain one, as is one into memory of the
// runtime's own and one below MIN_STAGED: 6 MB gain 0.1 ms at most.
//
// A copy leaves nothing behind on the caller's stream, and no mapping of the
// process changes.  A handle's stream is destroyed with it, and the next
// handle's is as good as free where the runtime has that queue ready again;
// where it has not (the same times come where streams are never destroyed),
// a new queue costs 1.1 ms and its first uploads run at 2.6 GB/s.  With the DMAs on the caller's stream, or with
// default-size stacks for eight threads (64 MB, more than the C library keeps
// for reuse, so that every copy unmapped some), that met most handles made
// after one was read and destroyed; making the lane again cost as much.  For a
// handle made, stepped twice, read and destroyed, ms (plain copies; as it was;
// now): 9 MB 1.4, 8.6, 1.3; 20 MB 3.0, 11, 2.4; 54 MB 7.9, 12, 6.5.  So one lane
// also outlives the last handle, and is freed when a later last handle goes
// without one of its generation having needed it.
#include <hip/hip_runtime.h>
#include <pthread.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "sfv_transfer.hpp"

namespace sfv {
namespace {

constexpr int SLOTS = 8, MAX_LANES = 4, MAX_WORKERS = 8;
constexpr size_t SLOT_BYTES = (size_t)2 << 20;
constexpr size_t MIN_STAGED = (size_t)8 << 20;
constexpr size_t WORKER_STACK = (size_t)256 << 10;

struct Lane {
    int device = -1;                    // -1: not made yet
    bool busy = false;
    hipStream_t stream = nullptr;
    // pinned, SLOTS slots of SLOT_BYTES, in one allocation made by the first copy
    // (eight allocations and their release took 2 ms each)
    char* memory = nullptr;
    hipEvent_t arrived[SLOTS] = {};
    char* slot(long c) const { return memory + (size_t)(c % SLOTS) * SLOT_BYTES; }
    // false if memory is short
    bool reserve() {
        if (!stream && hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess) {
            stream = nullptr;
            (void)hipGetLastError();
            return false;
        }
        if (!memory && hipHostMalloc((void**)&memory, SLOTS * SLOT_BYTES, hipHostMallocDefault) != hipSuccess) {
            memory = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (hipEvent_t& e : arrived)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                (void)hipGetLastError();
                return false;
            }
        return true;
    }
    void release() {
        if (memory) (void)hipHostFree(memory);
        memory = nullptr;
        for (hipEvent_t& e : arrived) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
        device = -1;
    }
};

std::mutex g_mu;
Lane g_lanes[MAX_LANES];
int g_users = 0;
bool g_needed = false;                  // a lane was taken since the first of these users came

// A free lane of this device (an event serves its own device's streams only),
// or nullptr.
Lane* take_lane(int device) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_needed = true;
    for (Lane& l : g_lanes)
        if (!l.busy && l.device == device) {
            l.busy = true;
            return &l;
        }
    for (Lane& l : g_lanes)
        if (!l.busy && l.device < 0) {
            l.busy = true;
            l.device = device;
            return &l;
        }
    return nullptr;
}
void give_lane(Lane* l) {
    std::lock_guard<std::mutex> lk(g_mu);
    l->busy = false;
}

hipError_t plain(void* dst, const void* src, size_t n, hipStream_t st) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st);
    const hipError_t s = hipStreamSynchronize(st);
    return e != hipSuccess ? e : s;
}

// Memory the runtime allocated (pinned, managed or device): it writes that
// itself, at the DMA's rate, and a host thread may not even have access to it.
// Through the slots a pinned 35 MB took 950 us, written by the runtime 620.
bool runtime_memory(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

// Chunk c travels through slot c mod SLOTS.  `arrived` counts the chunks whose
// DMA has completed, emptied[s] those copied out of slot s.
hipError_t staged(Lane& L, char* dst, const char* src, size_t n, size_t chunk, int want) {
    const hipStream_t st = L.stream;
    const long chunks = (long)((n + chunk - 1) / chunk);
    std::atomic<long> arrived{0}, next{0};
    std::atomic<bool> stop{false};
    std::atomic<long> emptied[SLOTS];
    for (auto& e : emptied) e.store(0);
    auto bytes = [&](long c) { return std::min(chunk, n - (size_t)c * chunk); };
    auto empty_slot = [&](long c) {
        std::memcpy(dst + (size_t)c * chunk, L.slot(c), bytes(c));
        emptied[c % SLOTS].store(c / SLOTS + 1, std::memory_order_release);
    };
    auto work = [&] {
        for (;;) {
            const long c = next.fetch_add(1);
            if (c >= chunks) return;
            while (arrived.load(std::memory_order_acquire) <= c) {
                if (stop.load()) return;
                std::this_thread::yield();
            }
            empty_slot(c);
        }
    };
    auto slot_free = [&](long c) { return emptied[c % SLOTS].load(std::memory_order_acquire) >= c / SLOTS; };
    hipError_t e = hipSuccess;
    long queued = 0;
    auto queue = [&] {
        const int s = (int)(queued % SLOTS);
        e = hipMemcpyAsync(L.slot(queued), src + (size_t)queued * chunk, bytes(queued), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(L.arrived[s], st);
        ++queued;
    };
    while (e == hipSuccess && queued < chunks && queued < SLOTS) queue();
    pthread_t workers[MAX_WORKERS];
    int running = 0;
    auto entry = [](void* w) -> void* {
        (*static_cast<decltype(work)*>(w))();
        return nullptr;
    };
    pthread_attr_t attr;
    if (pthread_attr_init(&attr) == 0) {
        (void)pthread_attr_setstacksize(&attr, WORKER_STACK);
        // no more threads: those there are, or this one, do it
        while (e == hipSuccess && running < want && pthread_create(&workers[running], &attr, entry, &work) == 0) ++running;
        (void)pthread_attr_destroy(&attr);
    }
    for (long c = 0; c < chunks && e == hipSuccess; ++c) {
        e = hipEventSynchronize(L.arrived[c % SLOTS]);
        if (e != hipSuccess) break;
        if (running) arrived.store(c + 1, std::memory_order_release);
        else empty_slot(c);
        while (e == hipSuccess && queued < chunks && slot_free(queued)) queue();
        // nothing under way: the next chunk's slot must be emptied first
        while (e == hipSuccess && queued == c + 1 && queued < chunks) {
            if (slot_free(queued)) queue();
            else std::this_thread::yield();
        }
    }
    if (e != hipSuccess) {
        stop.store(true);
        (void)hipStreamSynchronize(st);  // no DMA into a slot outlives the copy
    }
    for (int k = 0; k < running; ++k) (void)pthread_join(workers[k], nullptr);
    return e;
}

}  // namespace

void staging_retain() {
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_users;
}
void staging_release() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_users > 0) return;
    bool keep = g_needed;               // one, for the next user
    g_needed = false;
    for (Lane& l : g_lanes) {
        if (l.busy) continue;
        if (keep && l.memory) keep = false;
        else l.release();
    }
}

int staging_lanes() {
    std::lock_guard<std::mutex> lk(g_mu);
    int n = 0;
    for (const Lane& l : g_lanes) n += l.memory != nullptr;
    return n;
}

hipError_t copy_to_host(void* dst, const void* src, size_t n, hipStream_t st) {
    int device = 0;
    if (n < MIN_STAGED || hipGetDevice(&device) != hipSuccess || runtime_memory(dst)) return plain(dst, src, n, st);
    Lane* lane = take_lane(device);
    if (!lane) return plain(dst, src, n, st);
    // at least eight chunks, of at most a slot
    const size_t chunk = std::min(SLOT_BYTES, (n + SLOTS - 1) / SLOTS);
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
    // a worker for every slot's worth: starting one takes 15 us, copying 2 MB 200
    const int want = (int)std::min({(long)(n / SLOT_BYTES), (long)MAX_WORKERS, (long)std::max(1, cpus / 2)});
    hipError_t e;
    if (lane->reserve()) {
        e = hipStreamSynchronize(st);
        if (e == hipSuccess) e = staged(*lane, (char*)dst, (const char*)src, n, chunk, want);
    } else {
        e = plain(dst, src, n, st);
    }
    give_lane(lane);
    return e;
}

}  // namespace sfv
