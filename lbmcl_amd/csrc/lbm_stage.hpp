// lbm_stage.hpp -- blocking copies from device memory into a caller's memory: where
// it is pageable, through pinned staging buffers.
//
// hipMemcpy into pageable memory moves 10 GB/s on MI355X (the runtime copies
// through its own staging on one thread, which also takes the page faults of a
// fresh destination); the link moves 56 GB/s into pinned memory.  Here the bytes
// go in chunks through pinned buffers, and above kThreadsAbove a few threads copy
// the chunks that have arrived while the next ones are on the link.  Measured, 1
// GiB into fresh pages: 101 ms with hipMemcpy, 75 / 42 / 27 / 25 / 24 ms with 1 / 2
// / 4 / 6 / 8 threads and chunks of 4 MiB; 4 KiB 22 us with hipMemcpy, 12 us here.
// Memory that the device reaches itself (a caller's pinned buffer) takes the link's
// copy without a detour: 1.28 GB in 27.0 ms staged, 22.3 straight; asking the
// runtime what the pointer is takes a microsecond.
// The other direction stays with hipMemcpy: its source's pages exist, and it
// reads them at 25 GB/s (25 MB in 1.0 ms, 4.5 ms this way).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>

#include "lbm_pool.hpp"

namespace lbm_host {

// The process's pinned buffers, at most HostStage::kBuffers * kChunk (32 MiB),
// allocated by the first copies that need them (0.3 to 4 ms, so not for every
// context) and given back by lbm_trim.  One copy uses them at a time; another
// thread's goes the runtime's way meanwhile.
struct PinnedBuffers {
    std::mutex busy;  // held for the whole of a copy
    char* data = nullptr;
    size_t capacity = 0;

    hipError_t reserve(size_t bytes) {
        if (bytes <= capacity) return hipSuccess;
        free();
        void* p = nullptr;
        const hipError_t rc = hipHostMalloc(&p, bytes, hipHostMallocPortable);
        if (rc != hipSuccess) return rc;
        data = static_cast<char*>(p);
        capacity = bytes;
        return hipSuccess;
    }
    void free() {
        if (data) (void)hipHostFree(data);
        data = nullptr;
        capacity = 0;
    }
};
inline PinnedBuffers g_pinned;

// Copies of one context, whose events they use.  A context serves one host
// thread at a time.
struct HostStage {
    static constexpr int kBuffers = 8;
    static constexpr int kThreads = 4;
    static constexpr size_t kChunk = size_t(4) << 20;
    static constexpr size_t kThreadsAbove = size_t(2) << 20;

    hipEvent_t landed[kBuffers] = {};  // the copy into a buffer is done

    void release() {
        for (hipEvent_t& e : landed) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    hipError_t create_events() {
        for (hipEvent_t& e : landed) {
            if (e) continue;
            const hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
            if (rc != hipSuccess) {
                e = nullptr;
                return rc;
            }
        }
        return hipSuccess;
    }

    // Whether the device writes to the caller's memory without a staging buffer.
    static bool reached(const void* host) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return false;
    }

    // Copy `bytes` of `dev` into `host` behind the work enqueued on `stream`;
    // returns with the bytes in place.  `enqueued` is called once, when every copy
    // is on the stream.
    template <class F>
    hipError_t copy(int device, hipStream_t stream, void* host, const void* dev, size_t bytes, F&& enqueued) {
        const size_t chunk = bytes <= kThreadsAbove ? kChunk / 16 : bytes <= 4 * kChunk ? kChunk / 4 : kChunk;
        const int64_t chunks = int64_t((bytes + chunk - 1) / chunk);
        std::unique_lock<std::mutex> lock(g_pinned.busy, std::defer_lock);
        if (reached(host) || !lock.try_lock() || create_events() != hipSuccess ||
            g_pinned.reserve(kBuffers * (bytes <= kThreadsAbove ? kChunk / 16 : kChunk)) != hipSuccess) {
            (void)hipGetLastError();  // no need of pinned buffers, or none: as the runtime does it
            const hipError_t rc = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
            enqueued();
            const hipError_t rs = hipStreamSynchronize(stream);
            return rc != hipSuccess ? rc : rs;
        }
        char* const to = static_cast<char*>(host);
        const char* const from = static_cast<const char*>(dev);
        const auto size_of = [&](int64_t i) { return std::min(chunk, bytes - size_t(i) * chunk); };
        const auto buffer = [&](int64_t i) { return g_pinned.data + size_t(i % kBuffers) * chunk; };

        // Per buffer: the last chunk whose copy is enqueued, and the last one taken
        // out.  A buffer's next copy is enqueued after its last chunk was taken out,
        // and only then is its event recorded again.
        std::atomic<int64_t> sent[kBuffers], taken[kBuffers];
        for (int b = 0; b < kBuffers; ++b) {
            sent[b].store(-1);
            taken[b].store(-1);
        }
        std::atomic<int> failed{int(hipSuccess)};
        const auto good = [&] { return failed.load(std::memory_order_relaxed) == int(hipSuccess); };
        const auto wait_for = [&](const std::atomic<int64_t>& v, int64_t i) {
            while (v.load(std::memory_order_acquire) < i && good()) std::this_thread::yield();
            return good();
        };
        int64_t next = 0;  // the next chunk to enqueue
        const auto send_next = [&] {
            const int b = int(next % kBuffers);
            hipError_t e = hipMemcpyAsync(buffer(next), from + size_t(next) * chunk, size_of(next), hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(landed[b], stream);
            if (e != hipSuccess) failed.store(int(e));
            else sent[b].store(next++, std::memory_order_release);
            if (e == hipSuccess && next == chunks) enqueued();
        };
        const auto take = [&](int64_t i) {
            const int b = int(i % kBuffers);
            if (!wait_for(sent[b], i)) return;
            const hipError_t e = hipEventSynchronize(landed[b]);
            if (e != hipSuccess) {
                failed.store(int(e));
                return;
            }
            std::memcpy(to + size_t(i) * chunk, buffer(i), size_of(i));
            taken[b].store(i, std::memory_order_release);
        };

        // the link starts first, and no thread spins while the stream is busy with what is before it
        while (next < std::min<int64_t>(kBuffers, chunks) && good()) send_next();
        if (good()) {
            const hipError_t e = hipEventSynchronize(landed[0]);
            if (e != hipSuccess) failed.store(int(e));
        }
        std::thread threads[kThreads];
        int running = 0;
        const int wanted = bytes > kThreadsAbove ? int(std::min<int64_t>(kThreads, chunks)) : 0;
        std::atomic<int64_t> ticket{0};  // chunks are taken in order
        const auto work = [&] {
            (void)hipSetDevice(device);
            for (int64_t i = ticket.fetch_add(1); i < chunks && good(); i = ticket.fetch_add(1)) take(i);
        };
        for (; running < wanted; ++running) {
            try {
                threads[running] = std::thread(work);
            } catch (...) {
                break;  // as many as there are; none: this thread does the work
            }
        }
        if (running > 0) {
            while (next < chunks && good() && wait_for(taken[next % kBuffers], next - kBuffers)) send_next();
        } else {
            for (int64_t i = 0; i < chunks && good(); ++i) {
                take(i);
                if (next < chunks && good()) send_next();
            }
        }
        for (int t = 0; t < running; ++t) threads[t].join();
        if (good()) return hipSuccess;  // every copy was waited for
        (void)hipStreamSynchronize(stream);
        return hipError_t(failed.load());
    }
};

}  // namespace lbm_host
