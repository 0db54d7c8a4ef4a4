// lbm_pool.hpp -- device memory kept for the next context or gradient.
//
// hipMalloc and hipFree of a gradient's states cost more than the gradient: the
// driver clears memory that was freed before it hands it out again, at about 60
// GB/s, so a program that computes one gradient after another waits for that.
// Measured on several hosts, which differ in how long the driver takes, calls one
// after another without the pool / with it: 256^3 FP32 x 200 (40 GB of states, 310
// ms of kernels) 376 to 1008 ms / 320; 64^3 FP64 x 150 17.3 to 17.9 / 7.4, with a
// tape of all states.  The first call of a process has no pool yet: 393 / 334 and
// 27.4 / 22.6 (other memory, and the tapes).  Freed blocks are kept
// here and given out again by their exact size, which is that of a state for any
// number of steps.
//
// Bounds: a block of at most kBlockShare of the device's memory, all of them
// together at most kShare of it and (beyond kSmallShare) what else is free of it,
// kMax blocks;
// beyond that the ones kept longest are freed.  lbm_trim frees all, and what
// contexts keep for themselves between their calls (g_spares), and so does an
// allocation of this library that finds no memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace lbm_host {

// For the calling thread: an allocation is allowed while somebody records a HIP
// graph on a stream of their own, which forbids it to all threads by default and
// is broken by one.  For allocations in calls that otherwise only launch; those that
// wait for a stream (reads, lbm_finish) the runtime refuses then in any case.
struct AllowAllocation {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    AllowAllocation() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~AllowAllocation() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    AllowAllocation(const AllowAllocation&) = delete;
    AllowAllocation& operator=(const AllowAllocation&) = delete;
};

class DevicePool {
public:
    static constexpr size_t kBlockShare = 64;

    // A block of exactly `bytes` of the device, or null.
    void* take(int device, size_t bytes) {
        std::lock_guard<std::mutex> lock(mu_);
        for (int k = count_ - 1; k >= 0; --k) {
            if (blocks_[k].device != device || blocks_[k].bytes != bytes) continue;
            void* const p = blocks_[k].p;
            remove(k);
            return p;
        }
        return nullptr;
    }

    // Keep or free a block of the current device that no enqueued work uses.
    void give(int device, void* p, size_t bytes) {
        if (!p) return;
        std::lock_guard<std::mutex> lock(mu_);
        ask_total();
        if (bytes > total_ / kBlockShare) {
            (void)hipFree(p);
            return;
        }
        size_t held = bytes + sum(device);
        for (int k = 0; k < count_ && held > total_ / kShare;) {
            if (blocks_[k].device != device) {
                ++k;
                continue;
            }
            held -= blocks_[k].bytes;
            (void)hipFree(blocks_[k].p);
            remove(k);
        }
        if (count_ == kMax) {
            (void)hipFree(blocks_[0].p);
            remove(0);
        }
        blocks_[count_++] = Block{p, bytes, device};
    }

    // After a give, or several: leave at least as much free as is kept, for other
    // allocators of the process, which cannot ask for any of this.  Less than
    // 1/kSmallShare (1.2 GB) is not worth the question (5 us, of a small gradient's
    // 1.3 ms).
    void leave_half(int device) {
        std::lock_guard<std::mutex> lock(mu_);
        size_t held = sum(device), free_bytes = 0, total = 0;
        if (held <= total_ / kSmallShare) return;
        if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        for (int k = 0; k < count_ && held > free_bytes;) {
            if (blocks_[k].device != device) {
                ++k;
                continue;
            }
            held -= blocks_[k].bytes;
            free_bytes += blocks_[k].bytes;
            (void)hipFree(blocks_[k].p);
            remove(k);
        }
    }

    // Bytes kept of the device.
    size_t held(int device) {
        std::lock_guard<std::mutex> lock(mu_);
        return sum(device);
    }

    // The memory of a device (0: unknown).
    size_t device_memory() {
        std::lock_guard<std::mutex> lock(mu_);
        ask_total();
        return total_;
    }

    // Free everything; whether there was anything.
    bool trim() {
        std::lock_guard<std::mutex> lock(mu_);
        const bool any = count_ > 0;
        for (int k = 0; k < count_; ++k) (void)hipFree(blocks_[k].p);
        count_ = 0;
        return any;
    }

private:
    static constexpr int kMax = 512;
    static constexpr size_t kShare = 4;
    static constexpr size_t kSmallShare = 256;
    struct Block {
        void* p;
        size_t bytes;
        int device;
    };
    void ask_total() {  // of the first device used; the others are alike
        size_t free_bytes = 0;
        if (total_ == 0 && hipMemGetInfo(&free_bytes, &total_) != hipSuccess) {
            (void)hipGetLastError();
            total_ = 0;
        }
    }
    size_t sum(int device) const {
        size_t s = 0;
        for (int k = 0; k < count_; ++k) s += blocks_[k].device == device ? blocks_[k].bytes : 0;
        return s;
    }
    void remove(int k) {  // in order of age
        for (int j = k + 1; j < count_; ++j) blocks_[j - 1] = blocks_[j];
        --count_;
    }

    std::mutex mu_;
    Block blocks_[kMax];
    int count_ = 0;
    size_t total_ = 0;  // the device's memory
};
inline DevicePool g_pool;

// Memory that a context keeps between its calls, and that anybody in need may take
// from it there: an entry is in the list while it is parked.
struct Spare {
    void* p = nullptr;
    hipStream_t stream = nullptr;  // the work that uses it
    Spare *next = nullptr, *prev = nullptr;
};
class SpareList {
public:
    void park(Spare& s, void* p, hipStream_t stream) {
        if (!p) return;
        std::lock_guard<std::mutex> lock(mu_);
        s.p = p;
        s.stream = stream;
        s.prev = nullptr;
        s.next = head_;
        if (head_) head_->prev = &s;
        head_ = &s;
    }
    // What was parked, for the context alone again; null if somebody took it.
    void* take(Spare& s) {
        std::lock_guard<std::mutex> lock(mu_);
        void* const p = s.p;
        if (p) remove(s);
        return p;
    }
    // Free everything parked; whether there was anything.
    bool trim() {
        std::lock_guard<std::mutex> lock(mu_);
        const bool any = head_ != nullptr;
        while (head_) {
            (void)hipStreamSynchronize(head_->stream);
            (void)hipFree(head_->p);
            remove(*head_);
        }
        return any;
    }

private:
    void remove(Spare& s) {
        if (s.prev) s.prev->next = s.next;
        else head_ = s.next;
        if (s.next) s.next->prev = s.prev;
        s.p = nullptr;
    }
    std::mutex mu_;
    Spare* head_ = nullptr;
};
inline SpareList g_spares;

// Free what is kept; whether there was anything.
inline bool reclaim_memory() {
    const bool pool = g_pool.trim(), spares = g_spares.trim();
    return pool || spares;
}

}  // namespace lbm_host
