// lbm_small.hip -- several iterations of a small lattice in one launch: the rule
// that selects it, and the launches of every form but LBM_ARITH_OPENCL.
#include "lbm_range.hpp"
#include "lbm_small_launch.hpp"

namespace lbm_host {

bool small_is_one_tile(const StepPlan* c) { return c->n <= 8; }

// A launch of a lattice of one tile is bounded: about a millisecond.
constexpr int32_t kOneTileSteps = 1000;

int32_t small_steps(const StepPlan* c) {
    if (c->cfg.kernel != LBM_KERNEL_AUTO || c->n < 4) return 0;
    if (small_is_one_tile(c)) return kOneTileSteps;
    if (c->n == 16) return SmallTile16::G + 1;
    if (c->n == 32) return SmallTile32::G + 1;
    return 0;
}
int launch_small(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase) {
    using namespace lbm;
    switch (arith_of(c)) {
        case AR_OPENCL: return launch_small_opencl(c, src, dst, prev, k, every, phase);
        case AR_FUSED:
            return c->cfg.precision == LBM_F64 ? launch_small_impl<double, ST_NATIVE, AR_FUSED>(c, src, dst, prev, k, every, phase)
                                               : launch_small_impl<float, ST_NATIVE, AR_FUSED>(c, src, dst, prev, k, every, phase);
        case AR_EXACT:
            return c->cfg.precision == LBM_F64 ? launch_small_impl<double, ST_NATIVE, AR_EXACT>(c, src, dst, prev, k, every, phase)
                                               : launch_small_impl<float, ST_NATIVE, AR_EXACT>(c, src, dst, prev, k, every, phase);
        default:
            return c->cfg.storage == LBM_STORE_FP16_SHIFT
                       ? launch_small_impl<float, ST_FP16, AR_DELTA>(c, src, dst, prev, k, every, phase)
                       : launch_small_impl<float, ST_BF16, AR_DELTA>(c, src, dst, prev, k, every, phase);
    }
}

}  // namespace lbm_host
