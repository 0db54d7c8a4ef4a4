// tapes_test.cpp -- a gradient's device memory (lbmcl_amd/csrc/lbm_tapes.hpp) from an
// allocator with a given capacity: it succeeds exactly where what it cannot do
// without fits, whatever the optional tapes find; those come last, in whole
// segments, and an unfinished one is given back.  Exit status 0 when every check passes.
#include <cstdio>
#include <cstdlib>

#include "lbm_tapes.hpp"

namespace {

int failures = 0;
void check(bool ok, const char* what, long a, long b) {
    if (!ok) {
        std::fprintf(stderr, "FAIL %s (%ld, %ld)\n", what, a, b);
        ++failures;
    }
}

struct Device {
    size_t capacity, device, blocks_to_failure = SIZE_MAX;  // what is free, the device's memory
    size_t reported = 0;                                     // what available() says beyond the truth
    std::vector<std::pair<void*, size_t>> blocks;
    size_t used = 0, optional = 0;
    bool take(void** p, size_t bytes) {
        if (used + bytes > capacity || blocks.size() >= blocks_to_failure) return false;
        *p = std::malloc(1);
        blocks.emplace_back(*p, bytes);
        used += bytes;
        return true;
    }
    int alloc(void** p, size_t bytes, const char*) {
        check(optional == 0, "what is needed comes before what is optional", long(blocks.size()), 0);
        return take(p, bytes) ? 0 : -3;
    }
    bool try_alloc(void** p, size_t bytes) {
        const bool ok = take(p, bytes);
        optional += ok ? 1 : 0;
        return ok;
    }
    void give_back(size_t n) {
        for (; n > 0; --n) {
            std::free(blocks.back().first);
            used -= blocks.back().second;
            blocks.pop_back();
            --optional;
        }
    }
    size_t available() const { return capacity - used + reported; }
    size_t total() const { return device; }
    ~Device() {
        for (const auto& b : blocks) std::free(b.first);
    }
};

void run(const lbm_host::GradientSizes& z, size_t capacity, size_t device, size_t reported, size_t blocks) {
    Device d{capacity, device, blocks, reported, {}, 0, 0};
    lbm_host::GradientMemory m;
    const int rc = allocate_gradient(d, z, &m);
    const size_t needed_blocks = size_t(z.segments - 1 + z.tape + 2 + (z.grad ? 1 : 0) + (z.grad_stage ? 1 : 0) + 2);
    const size_t needed = size_t(z.segments - 1 + z.tape + 2) * z.state + z.grad + z.grad_stage + z.partials + z.sums;
    check(needed_bytes(z) == double(needed), "needed bytes", long(needed), 0);
    check((rc == 0) == (needed <= capacity && needed_blocks <= blocks), "succeeds where the needed memory fits", long(capacity),
          long(blocks));
    if (rc) return;
    check(m.kept >= 1 && m.kept <= z.segments, "segments kept", long(m.kept), long(z.segments));
    check(m.tapes.size() == size_t(m.kept * z.tape), "whole tapes", long(m.tapes.size()), long(m.kept));
    for (void* p : m.tapes) check(p != nullptr, "a tape's state", long(capacity), 0);
    for (void* p : m.checkpoints) check(p != nullptr, "a checkpoint", long(capacity), 0);
    check(m.lambda[0] && m.lambda[1] && m.partials && m.sums, "needed blocks", long(capacity), 0);
    check((m.grad != nullptr) == (z.grad > 0) && (m.grad_stage != nullptr) == (z.grad_stage > 0), "gradient", 0, 0);
    const size_t extra = size_t((m.kept - 1) * z.tape);
    check(d.optional == extra && d.used == needed + extra * z.state, "nothing else is held", long(d.used), long(extra));
    if (reported == 0 && extra > 0) {
        check(extra * z.state <= (capacity - needed) / 2, "half of what is left stays", long(capacity), long(extra));
        check(2 * z.state + d.used <= device / 16, "a sixteenth of the device's memory", long(d.used), long(device));
    }
    check(z.extra || extra == 0, "no tapes that nobody wants", long(extra), 0);
    if (z.extra && z.tape > 0 && reported == 0 && blocks == SIZE_MAX && m.kept < z.segments) {  // another one would not do
        const size_t more = (extra + size_t(z.tape)) * z.state;
        check(more > (capacity - needed) / 2 || 2 * z.state + needed + more > device / 16, "as many as there is room for",
              long(capacity), long(extra));
    }
}

}  // namespace

int main() {
    for (const int64_t segments : {1, 2, 3, 13})
        for (const int64_t tape : {0, 1, 4, 11})
            for (const int grad : {0, 1, 2, 3}) {
                lbm_host::GradientSizes z;
                z.segments = segments;
                z.tape = tape;
                z.state = 1000;
                z.extra = grad < 3;
                z.grad = grad > 0 ? 160 : 0;
                z.grad_stage = grad > 1 ? 80 : 0;
                z.partials = 48;
                z.sums = 24;
                for (const size_t device : {size_t(64) << 10, size_t(400) << 10, size_t(1) << 30}) {
                    for (size_t capacity = 0; capacity < 400000; capacity += 997) run(z, capacity, device, 0, SIZE_MAX);
                    for (size_t blocks = 0; blocks < 180; ++blocks) run(z, size_t(1) << 30, device, 0, blocks);
                    // memory that others take after the question
                    for (size_t capacity = 0; capacity < 200000; capacity += 4999)
                        run(z, capacity, device, size_t(1) << 28, SIZE_MAX);
                }
            }
    if (failures) return 1;
    std::printf("all checks passed\n");
    return 0;
}
