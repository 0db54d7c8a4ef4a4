// lbm_tapes.hpp -- the device memory of a gradient: first all that it cannot do
// without, then tapes that save it time.  Host code without HIP: the allocator is
// the caller's.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace lbm_host {

struct GradientSizes {
    int64_t segments = 0;      // checkpoints, the first of which is the context's lattice
    int64_t tape = 0;          // states of a segment's tape
    size_t state = 0;          // bytes of a state
    size_t grad = 0;           // of the body force's gradient (0: not wanted)
    size_t grad_stage = 0;     // of what it is accumulated in (0: in itself)
    size_t partials = 0, sums = 0;
    bool extra = true;         // tapes beyond what is needed are wanted
};

struct GradientMemory {
    std::vector<void*> checkpoints;  // segments 1, 2, ...
    std::vector<void*> tapes;        // the last segment's, then those of the segments before it
    int64_t kept = 0;                // segments whose states stay on a tape of their own
    void* lambda[2] = {nullptr, nullptr};
    void *grad = nullptr, *grad_stage = nullptr, *partials = nullptr, *sums = nullptr;
};

// What the gradient cannot do without, in floating point: it may be more than any
// device has.
inline double needed_bytes(const GradientSizes& z) {
    return (double(z.segments - 1) + double(z.tape) + 2.0) * double(z.state) +
           double(z.grad + z.grad_stage + z.partials + z.sums);
}

// Tapes beyond the last segment's.  Each saves the recomputation of its states,
// which otherwise is a second forward run.  A caller who chose the interval of the
// checkpoints chose the memory with it and gets none.  They are for plentiful memory: with all
// that the gradient holds (`held`, the context's lattices too) they fit a sixteenth
// of the device's (18 GB: all of 64^3 FP64 x 150 in 6 GB, 128^3 FP32 up to 110
// steps), and they leave half of what is left to others.
inline int64_t extra_tapes(const GradientSizes& z, size_t held, size_t available, size_t total) {
    if (!z.extra || z.tape == 0) return 0;  // segments of one step need none
    const size_t share = total / 16 > held ? total / 16 - held : 0;
    const size_t room = std::min(share, available / 2);
    return std::min<int64_t>(z.segments - 1, int64_t(room / (size_t(z.tape) * z.state)));
}

// A has: int alloc(void**, size_t, const char*), which returns 0 or an error's
// code; bool try_alloc(void**, size_t); give_back(n), the n blocks allocated last;
// and available() and total(), bytes of the device.
template <class A> int allocate_gradient(A& a, const GradientSizes& z, GradientMemory* m) {
    size_t held = 2 * z.state;  // the context's lattices
    const auto needed = [&](void** p, size_t bytes, const char* what) {
        held += bytes;
        return a.alloc(p, bytes, what);
    };
    int rc = 0;
    m->checkpoints.assign(size_t(z.segments - 1), nullptr);
    for (size_t k = 0; k < m->checkpoints.size() && !rc; ++k) rc = needed(&m->checkpoints[k], z.state, "adjoint checkpoint");
    m->tapes.assign(size_t(z.tape), nullptr);
    for (size_t k = 0; k < m->tapes.size() && !rc; ++k) rc = needed(&m->tapes[k], z.state, "adjoint tape");
    for (int j = 0; j < 2 && !rc; ++j) rc = needed(&m->lambda[j], z.state, "adjoint state");
    if (!rc && z.grad) rc = needed(&m->grad, z.grad, "dJ/dg");
    if (!rc && z.grad_stage) rc = needed(&m->grad_stage, z.grad_stage, "dJ/dg accumulator");
    if (!rc) rc = needed(&m->partials, z.partials, "partials");
    if (!rc) rc = needed(&m->sums, z.sums, "accumulators");
    if (rc) return rc;
    m->kept = 1;
    const size_t available = z.extra && z.tape > 0 ? a.available() : 0;  // before total()
    const int64_t extra = extra_tapes(z, held, available, a.total());
    m->tapes.reserve(size_t((1 + extra) * z.tape));
    while (m->kept < 1 + extra) {
        int64_t got = 0;
        for (void* p = nullptr; got < z.tape && a.try_alloc(&p, z.state); ++got) m->tapes.push_back(p);
        if (got < z.tape) {  // as many as there is memory for, and none of the unfinished one
            a.give_back(size_t(got));
            m->tapes.resize(size_t(m->kept * z.tape));
            break;
        }
        ++m->kept;
    }
    return 0;
}

}  // namespace lbm_host
