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

// lbm_relayout.hip: whether iterations are faster in the layout of stride
// kFastStride than in the plan's own (from 64^3 on: smaller lattices have their
// own kernel and are read through the caches whole), and a change of a lattice's
// layout.  Ranges of kRelayoutRange iterations or more are long against the three
// changes that they take: at 256^3 FP32 stride 16, where an iteration gains least
// against them, 3 x 0.55 ms against 32 x 0.11.
constexpr int64_t kFastStride = 4096, kRelayoutRange = 32;
bool relayout_pays(const StepPlan* c);
int relayout(lbm_ctx* c, const void* in, int64_t stride_in, void* out, int64_t stride_out);

}  // namespace lbm_host
