// lbm_range.hpp -- what lbm_compute_range has beyond single iterations: launches
// that take several, and another layout for the time of a range.
#pragma once

#include "lbm_ctx.hpp"

namespace lbm_host {

// lbm_small.hip: iterations per launch of a small lattice (0: none), and whether
// the lattice is one tile, whose launch leaves both lattices as single steps do.
// `phase`: number of the iteration before the first one, modulo `every`.
int32_t small_steps(const StepPlan* c);
bool small_is_one_tile(const StepPlan* c);
int launch_small(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase);

// lbm_relayout.hip: whether a range of `count` iterations is faster in the layout of
// stride kFastStride than in the plan's own, whether iterations are at all, and a
// change of a lattice's layout.
constexpr int64_t kFastStride = 4096;
bool relayout_possible(const StepPlan* c);
bool relayout_pays(const StepPlan* c, int64_t count);
// Whether a third lattice of that size, which a range can do without, may be
// allocated for one of `count` iterations: at most an eighth of the device's memory,
// and as much again stays free.  One too large for the pool is for ranges of 64
// iterations or more: the first one may have to wait for memory (10 GB at 512^3
// FP32, where an iteration gains 2 ms).
inline bool third_lattice_fits(size_t bytes, int64_t count, size_t free_bytes, size_t total) {
    return bytes <= total / (count < 64 ? DevicePool::kBlockShare : 8) && bytes <= free_bytes / 2;
}
int relayout(lbm_ctx* c, const void* in, int64_t stride_in, void* out, int64_t stride_out);

}  // namespace lbm_host
