// rules_test.cpp -- the rules by which a range of iterations is launched
// (lbmcl_amd/csrc/lbm_range.hpp), asked without a device: this program is host code
// alone and takes the library's functions from liblbm_hip.so.  Exit status 0 when
// every check passes.
#include "lbm_range.hpp"

using namespace lbm_host;

namespace {

int failures = 0;
void check(bool ok, const char* what, long a = 0, long b = 0, long c = 0) {
    if (!ok) {
        std::fprintf(stderr, "FAIL %s (%ld, %ld, %ld)\n", what, a, b, c);
        ++failures;
    }
}

// The third lattice: an eighth of the memory at most, for short ranges what the
// pool keeps, and never more than is free beside it.
void third_lattices() {
    const size_t G = size_t(1) << 30, total = 288 * G;
    check(third_lattice_fits(G, 12, 200 * G, total), "1 GB, much is free");
    check(third_lattice_fits(total / 64, 63, 200 * G, total), "the pool's largest block");
    check(!third_lattice_fits(total / 64 + 1, 63, 200 * G, total), "larger, for a short range");
    check(third_lattice_fits(total / 64 + 1, 64, 200 * G, total), "larger, for a long range");
    check(third_lattice_fits(36 * G, 64, 200 * G, total), "an eighth");
    check(!third_lattice_fits(36 * G + 1, 1000, 200 * G, total), "more than an eighth");
    check(third_lattice_fits(G, 64, 2 * G, total), "as much again is free");
    check(!third_lattice_fits(G, 64, 2 * G - 1, total), "less is free");
}

// Ranges that go through the other layout are at least as long as the measured
// number of iterations that pays for it (lbm_relayout.hip), and not much longer.
void other_layout() {
    struct Case {
        int precision, storage, n, stride;
        double pays_from;
    };
    const int f32 = LBM_F32, f64 = LBM_F64, own = LBM_STORE_NATIVE, h = LBM_STORE_FP16_SHIFT, b = LBM_STORE_BF16_SHIFT;
    for (const Case& k : {Case{f32, own, 64, 1, 9.5}, {f32, own, 64, 2, 10.3}, {f32, own, 64, 8, 7.9}, {f32, own, 64, 16, 7.3},
                          {f32, own, 128, 1, 8.3}, {f32, own, 128, 8, 7.7}, {f32, own, 128, 16, 19.6}, {f32, own, 256, 1, 8.8},
                          {f32, own, 256, 16, 28.2}, {f32, own, 512, 1, 9.2}, {f32, own, 512, 16, 14.9},
                          {f64, own, 64, 1, 6.6}, {f64, own, 64, 4, 5.8}, {f64, own, 64, 8, 59.6}, {f64, own, 128, 1, 11.1},
                          {f64, own, 128, 4, 10.6}, {f64, own, 128, 8, 55.4}, {f64, own, 256, 1, 8.8}, {f64, own, 256, 8, 44.2}, {f64, own, 512, 8, 77.0},
                          {f32, h, 64, 1, 20.1}, {f32, b, 64, 2, 17.3}, {f32, h, 64, 16, 13.5}, {f32, h, 64, 32, 13.3},
                          {f32, h, 128, 1, 4.5}, {f32, b, 128, 32, 4.1}, {f32, h, 256, 1, 6.2}, {f32, h, 256, 32, 9.7}}) {
        lbm_config c = LBM_CONFIG_INIT;
        c.dim = k.n;
        c.stride = k.stride;
        c.precision = k.precision;
        c.storage = k.storage;
        c.viscosity = 0.01;
        c.velocity = 0.05;
        StepPlan plan;
        check(plan_from_config(c, &plan) == LBM_OK, "a plan", k.n, k.stride);
        int64_t from = 1;
        while (from < 1000 && !relayout_pays(&plan, from)) ++from;
        check(from >= k.pays_from, "a range that does not pay for the other layout", k.n, k.stride, long(from));
        check(from <= 96, "a range that pays for the other layout", k.n, k.stride, long(from));
        c.kernel = LBM_KERNEL_GENERIC;
        check(plan_from_config(c, &plan) == LBM_OK && !relayout_pays(&plan, 1000), "a kernel of the caller's", k.n, k.stride);
    }
    for (const auto& k : {std::pair<int, int>{32, 1}, {128, 32}, {64, 64}, {512, 4096}}) {
        lbm_config c = LBM_CONFIG_INIT;
        c.dim = k.first;
        c.stride = k.second;
        c.viscosity = 0.01;
        c.velocity = 0.05;
        StepPlan plan;
        check(plan_from_config(c, &plan) == LBM_OK && !relayout_pays(&plan, 1 << 20), "stays in its layout", k.first, k.second);
    }
}

// A launch that no kernel was built for is an error, not a success without a launch
// (FP32 with a force, refused before the device is asked for anything).
void launches_without_a_kernel() {
    double force = 0;
    for (const int arith : {LBM_ARITH_OPENCL, LBM_ARITH_FUSED, LBM_ARITH_EXACT}) {
        lbm_config c = LBM_CONFIG_INIT;
        c.dim = 128;
        c.stride = 4096;
        c.viscosity = 0.01;
        c.velocity = 0.05;
        c.optimize = arith;
        StepPlan plan;
        check(plan_from_config(c, &plan) == LBM_OK && two_steps_preferred(&plan), "a plan for two steps", arith);
        plan.force = &force;
        check(!two_steps_preferred(&plan), "single steps with a force", arith);
        check(launch_two_steps(&plan, nullptr, nullptr, 0) == LBM_ERR_INVALID, "no two-step launch with a force", arith);
    }
}

}  // namespace

int main() {
    launches_without_a_kernel();
    other_layout();
    third_lattices();
    if (failures) return 1;
    std::printf("all checks passed\n");
    return 0;
}
