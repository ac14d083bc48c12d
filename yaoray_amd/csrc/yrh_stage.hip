// Large copies from the device to pageable host memory.
//
// What bounds them: a plain hipMemcpyAsync to pageable memory is staged by the
// runtime 1 MiB at a time on one thread, which also takes the page faults of a
// freshly allocated destination: 128 MiB take 7.6 ms, into a new array 13.0 ms,
// against 2.4 ms of the link. Here a few threads copy chunks through pinned
// buffers of the context: while one chunk is on the link, the same thread
// moves the one before it to the caller's memory (4.4 ms, new array or not).
// Copies to the device stay plain: 16 MiB take 0.46 ms that way and took 0.60 ms
// through the pinned buffers, 64 MiB 2.2 ms either way.
#include "yrh_internal.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <functional>
#include <new>
#include <thread>

namespace yrh {

namespace {

constexpr size_t kChunk = size_t{1} << 20;
constexpr int kMaxThreads = 8;  // the caller's among them
constexpr int kSlots = 2 * kMaxThreads;
// Below, starting threads costs what the copy gains (4 MiB: 45 us slower).
constexpr size_t kMinBytes = size_t{6} << 20;
// Chunks per thread that pay for starting one.
constexpr size_t kChunksPerThread = 2;

}  // namespace

struct HostStage {
    char* memory = nullptr;  // kSlots chunks, pinned
    hipEvent_t events[kSlots] = {};
    ~HostStage() {
        for (hipEvent_t e : events) {
            if (e != nullptr) (void)hipEventDestroy(e);
        }
        if (memory != nullptr) (void)hipHostFree(memory);
    }
};

void DestroyHostStage(yrh_context* ctx) {
    delete ctx->stage;
    ctx->stage = nullptr;
}

namespace {

// The context's device as the current one while in scope: events belong to the
// device that is current when they are made, and a copy leaves the caller's
// choice as it was.
struct DeviceScope {
    int before = -1;
    explicit DeviceScope(int device) {
        if (hipGetDevice(&before) != hipSuccess) before = -1;
        (void)hipSetDevice(device);
    }
    ~DeviceScope() {
        if (before >= 0) (void)hipSetDevice(before);
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;
};

// Whether the runtime knows nothing of p: pinned memory takes a plain copy at
// the speed of the link (128 MiB in 2.4 ms, 4.4 ms through these buffers), and
// device memory is not the host's to write.
bool Pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// The context's pinned buffers (16 MiB), or null: a context's first copy
// unless it pays for the allocation by itself (a context made for one frame
// reads one film; 32 MiB into a new array take 3.2 ms plainly, 1.3 ms through
// the buffers and 2.4 to 3.0 ms with their allocation, a process's first), or no
// memory to be had.
HostStage* Stage(yrh_context* ctx, size_t bytes) {
    if (ctx->stage != nullptr) return ctx->stage;
    if (!ctx->large_copy_seen && bytes < (size_t{32} << 20)) {
        ctx->large_copy_seen = true;
        return nullptr;
    }
    HostStage* s = new (std::nothrow) HostStage();
    if (s == nullptr) return nullptr;
    bool ok = hipHostMalloc(reinterpret_cast<void**>(&s->memory), kSlots * kChunk, hipHostMallocDefault) == hipSuccess;
    for (int k = 0; ok && k < kSlots; ++k) {
        ok = hipEventCreateWithFlags(&s->events[k], hipEventDisableTiming) == hipSuccess;
    }
    if (!ok) {
        (void)hipGetLastError();
        delete s;
        return nullptr;
    }
    ctx->stage = s;
    return s;
}

// Runs `work(k)` on as many threads as the copy fills, the caller's included.
template <class Work>
void RunThreads(size_t chunks, const Work& work) {
    const int threads = static_cast<int>(
        std::max<size_t>(1, std::min<size_t>(kMaxThreads, chunks / kChunksPerThread)));
    std::thread pool[kMaxThreads];
    try {
        for (int k = 1; k < threads; ++k) pool[k] = std::thread(std::cref(work), k);
    } catch (...) {  // no more threads, or no memory for one: the ones there take all chunks
    }
    work(0);
    for (std::thread& t : pool) {
        if (t.joinable()) t.join();
    }
}

}  // namespace

int StagedCopyToHost(yrh_context* ctx, void* dst, const void* src, size_t bytes, bool* done) {
    *done = false;
    if (bytes < kMinBytes || !Pageable(dst)) return YRH_OK;
    const DeviceScope scope(ctx->device);
    HostStage* s = Stage(ctx, bytes);
    if (s == nullptr) return YRH_OK;
    *done = true;
    const size_t chunks = (bytes + kChunk - 1) / kChunk;
    std::atomic<size_t> next{0};
    std::atomic<int> status{hipSuccess};
    auto work = [&](int thread) {
        if (thread != 0) (void)hipSetDevice(ctx->device);  // the caller's thread: done
        size_t held[2] = {chunks, chunks};  // the chunk in each of the thread's slots (chunks: none)
        for (int turn = 0;; turn ^= 1) {
            const int slot = 2 * thread + turn;
            const size_t c = status.load() == hipSuccess ? next.fetch_add(1) : chunks;
            held[turn] = c < chunks ? c : chunks;
            if (c < chunks) {
                const size_t at = c * kChunk;
                hipError_t e = hipMemcpyAsync(s->memory + static_cast<size_t>(slot) * kChunk,
                                              static_cast<const char*>(src) + at, std::min(kChunk, bytes - at),
                                              hipMemcpyDeviceToHost, ctx->stream);
                if (e == hipSuccess) e = hipEventRecord(s->events[slot], ctx->stream);
                if (e != hipSuccess) {
                    status.store(e);
                    held[turn] = chunks;
                }
            }
            // The chunk before it, meanwhile.
            const int other = turn ^ 1;
            if (held[other] < chunks) {
                const int oslot = 2 * thread + other;
                const hipError_t e = hipEventSynchronize(s->events[oslot]);
                if (e != hipSuccess) {
                    status.store(e);
                } else {
                    const size_t at = held[other] * kChunk;
                    std::memcpy(static_cast<char*>(dst) + at, s->memory + static_cast<size_t>(oslot) * kChunk,
                                std::min(kChunk, bytes - at));
                }
                held[other] = chunks;
            } else if (held[turn] == chunks) {
                return;
            }
        }
    };
    RunThreads(chunks, work);
    const hipError_t sync = hipStreamSynchronize(ctx->stream);
    const hipError_t e = static_cast<hipError_t>(status.load());
    return CheckHip(ctx, e != hipSuccess ? e : sync, "staged copy to host");
}

}  // namespace yrh
