// lbm_two_step.hip -- two iterations in one launch: the rule that selects it,
// and the launches of every form but LBM_ARITH_OPENCL.
#include "lbm_two_step_launch.hpp"

namespace lbm_host {

// Measured on MI355X against the single-step kernels (us per iteration, single /
// two-step):
//   lattice   128^3 FP32 48 / 36, FP64 95 / 69; at 64^3 FP32 8.4 / 13.9: too few
//             planes per block, so not below 128^3
//   stride    256^3 FP32: 32-byte runs (stride 8) 609 / 515, 16-byte ones 588 /
//             1143 (the lines of neighbouring populations are then fetched once for
//             each); FP64: 32-byte runs 1219 / 966, 16-byte ones 1180 / 3472
//   storage   256^3 FP16 218 / 285: bound by instructions, not by memory
//   force     256^3 FP32 424 / 485 (its registers do not fit), FP64 880 / 596
bool two_steps_possible(const StepPlan* c) {
    return c->cfg.kernel == LBM_KERNEL_AUTO && c->cfg.storage == LBM_STORE_NATIVE && c->n >= 128 &&
           c->stride * int64_t(c->ssize) >= 32;
}
bool two_steps_preferred(const StepPlan* c) { return two_steps_possible(c) && !(c->force && c->cfg.precision == LBM_F32); }

int launch_two_steps(StepPlan* c, const void* src, void* dst, int macro_last) {
    switch (arith_of(c)) {
        case lbm::AR_OPENCL: return launch_two_steps_opencl(c, src, dst, macro_last);
        case lbm::AR_FUSED:
            return c->cfg.precision == LBM_F64
                       ? launch_two_steps_impl<double, lbm::ST_NATIVE, lbm::AR_FUSED>(c, src, dst, macro_last)
                       : launch_two_steps_impl<float, lbm::ST_NATIVE, lbm::AR_FUSED>(c, src, dst, macro_last);
        case lbm::AR_EXACT:
            return c->cfg.precision == LBM_F64
                       ? launch_two_steps_impl<double, lbm::ST_NATIVE, lbm::AR_EXACT>(c, src, dst, macro_last)
                       : launch_two_steps_impl<float, lbm::ST_NATIVE, lbm::AR_EXACT>(c, src, dst, macro_last);
        default: return fail(LBM_ERR_INVALID, "16-bit storage has no two-step launch");
    }
}

}  // namespace lbm_host
