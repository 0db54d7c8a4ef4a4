// hip_runtime.h -- the few functions of the HIP runtime that the library's host-side
// headers use, on host memory, for tests without a device: a stream is a thread that
// does what is enqueued in order, "device" memory is malloc's, and calls can be made
// to fail.
#pragma once

#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;
struct hipPointerAttribute_t {
    hipMemoryType type;
};

namespace host_hip {

struct Stream {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> work;
    bool busy = false, end = false;
    std::thread thread{[this] {
        std::unique_lock<std::mutex> lock(mu);
        for (;;) {
            cv.wait(lock, [this] { return end || !work.empty(); });
            if (work.empty()) return;
            auto f = std::move(work.front());
            work.pop_front();
            busy = true;
            lock.unlock();
            f();
            lock.lock();
            busy = false;
            cv.notify_all();
        }
    }};
    void add(std::function<void()> f) {
        std::lock_guard<std::mutex> lock(mu);
        work.push_back(std::move(f));
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> lock(mu);
        cv.wait(lock, [this] { return work.empty() && !busy; });
    }
    ~Stream() {
        {
            std::lock_guard<std::mutex> lock(mu);
            end = true;
        }
        cv.notify_all();
        thread.join();
    }
};
struct Event {
    std::mutex mu;
    std::condition_variable cv;
    long recorded = 0, done = 0;
};

inline std::mutex mu;
inline std::map<const char*, size_t> pinned;  // what hipHostMalloc gave
inline long copies = 0, copies_to_fail = -1;  // enqueued so far; the one that fails
inline bool no_pinned_memory = false;

inline bool is_pinned(const void* p) {
    std::lock_guard<std::mutex> lock(mu);
    auto it = pinned.upper_bound(static_cast<const char*>(p));
    return it != pinned.begin() && (--it, static_cast<const char*>(p) < it->first + it->second);
}

}  // namespace host_hip

using hipStream_t = host_hip::Stream*;
using hipEvent_t = host_hip::Event*;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
inline hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = size_t(1) << 40;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (host_hip::no_pinned_memory) return hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    std::lock_guard<std::mutex> lock(host_hip::mu);
    host_hip::pinned[static_cast<char*>(*p)] = bytes;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lock(host_hip::mu);
    host_hip::pinned.erase(static_cast<char*>(p));
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = host_hip::is_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new host_hip::Event;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    {
        std::lock_guard<std::mutex> lock(e->mu);
        ++e->recorded;
    }
    s->add([e] {
        std::lock_guard<std::mutex> lock(e->mu);
        ++e->done;
        e->cv.notify_all();
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    std::unique_lock<std::mutex> lock(e->mu);
    const long want = e->recorded;
    e->cv.wait(lock, [e, want] { return e->done >= want; });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->wait();
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind, hipStream_t s) {
    if (host_hip::copies++ == host_hip::copies_to_fail) return hipErrorUnknown;
    s->add([=] { std::memcpy(to, from, bytes); });
    return hipSuccess;
}
