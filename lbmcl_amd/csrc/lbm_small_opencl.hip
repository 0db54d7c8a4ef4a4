// lbm_small_opencl.hip -- small-lattice launches in the LBM_ARITH_OPENCL form,
// built with OpenCL's FP32 division precision like lbm_opencl_arith.hip.
#include "lbm_small_launch.hpp"

namespace lbm_host {

int launch_small_opencl(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase) {
    return c->cfg.precision == LBM_F64
               ? launch_small_impl<double, lbm::ST_NATIVE, lbm::AR_OPENCL>(c, src, dst, prev, k, every, phase)
               : launch_small_impl<float, lbm::ST_NATIVE, lbm::AR_OPENCL>(c, src, dst, prev, k, every, phase);
}

}  // namespace lbm_host
