// lbm_two_step_opencl.hip -- two-step launches in the LBM_ARITH_OPENCL form,
// built with OpenCL's FP32 division precision like lbm_opencl_arith.hip.
#include "lbm_two_step_launch.hpp"

namespace lbm_host {

int launch_two_steps_opencl(StepPlan* c, const void* src, void* dst, int macro_last) {
    return c->cfg.precision == LBM_F64
               ? launch_two_steps_impl<double, lbm::ST_NATIVE, lbm::AR_OPENCL>(c, src, dst, macro_last)
               : launch_two_steps_impl<float, lbm::ST_NATIVE, lbm::AR_OPENCL>(c, src, dst, macro_last);
}

}  // namespace lbm_host
