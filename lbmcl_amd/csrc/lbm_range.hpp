// lbm_range.hpp -- launches that take more than one iteration, for
// lbm_compute_range.
#pragma once

#include "lbm_ctx.hpp"

namespace lbm_host {

// lbm_small.hip: iterations per launch of a small lattice (0: none), and whether
// the lattice is one tile, whose launch leaves both lattices as single steps do.
// `phase`: number of the iteration before the first one, modulo `every`.
int32_t small_steps(const StepPlan* c);
bool small_is_one_tile(const StepPlan* c);
int launch_small(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase);

}  // namespace lbm_host
