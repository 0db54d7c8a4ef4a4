// lbm_two_step_launch.hpp -- launching the two-step kernel, shared by the two
// translation units that instantiate it.
#pragma once

#include "lbm_ctx.hpp"
#include "lbm_two_step.hpp"

namespace lbm_host {

constexpr int64_t kTwoStepCUs = 256;  // MI355X; one block per CU

// Output planes per block.  A block spends a round per plane of its chunk and
// three more (the plane before the chunk, the one after it, and the first
// round's loads that nothing hides), and the launch takes as many turns as the
// blocks need on 256 CUs: the chunk length that minimises turns x rounds.
inline int64_t two_step_planes(int64_t n, int64_t tiles) {
    int64_t best = n - 2, cost = INT64_MAX;
    for (int64_t chunks = 1; chunks <= (n - 2 + 3) / 4; ++chunks) {
        const int64_t len = (n - 2 + chunks - 1) / chunks;
        const int64_t blocks = tiles * ((n - 2 + len - 1) / len);
        const int64_t c = ((blocks + kTwoStepCUs - 1) / kTwoStepCUs) * (len + 3);
        if (c < cost) {
            cost = c;
            best = len;
        }
    }
    return best;
}

// Columns of a tile's segment of a row.  The wider, the fewer lines of a row two
// tiles share and the longer the runs a block stores, but the fewer rows the
// block has threads for, of which it outputs all but two.  Measured (us per
// iteration, FP32 stride 4096, W = 64 / 128 / 256): 128^3 36.6 / 35.1 / -, 256^3
// 307 / 272 / 258, 512^3 2331 / 2192 / 2091; FP64 (W = 32 / 64 / 128): 128^3 75 / 68
// / 74, 256^3 596 / 545 / 517, 512^3 4889 / 4345 / 7290.  FP32 at 1024^3 needs more
// than two tiles in a row, hence halo threads, for which W = 256 leaves no rows.
template <class T> inline int32_t two_step_segment(int32_t n) {
    if (sizeof(T) == 4) return n <= 512 ? std::min(n, 256) : 128;
    return n == 256 ? 128 : 64;
}

template <class T, int KIND, int ARITH>
inline int launch_two_steps_impl(StepPlan* c, const void* src, void* dst, int macro_last) {
    if (sizeof(T) == 4 && c->force) return fail(LBM_ERR_INVALID, "no two-step launch in FP32 with a force");
    constexpr int threads = lbm::TwoStepThreads<T>::value;
    lbm::TwoStepArgs<T> a{};
    a.s = step_args<T, ARITH>(c, src, dst, 0, 0);
    a.macro_last = macro_last;
    a.w = two_step_segment<T>(c->n);
    a.tiles_x = c->n / a.w;
    a.halo = a.tiles_x > 2;
    a.rows = a.halo ? threads / (a.w + 2) : threads / a.w;
    a.tiles_y = (c->n - 2 + a.rows - 3) / (a.rows - 2);
    const int64_t tiles = int64_t(a.tiles_x) * a.tiles_y;
    a.zlen = int32_t(two_step_planes(c->n, tiles));
    const int64_t blocks = tiles * ((c->n - 2 + a.zlen - 1) / a.zlen);
    const dim3 grid{unsigned(blocks)}, block(threads);
    const bool contig = c->stride >= c->n;
    const auto launch = [&](auto kernel) { launch_on(c, kernel, grid, block, nullptr, nullptr, a); };
    if constexpr (sizeof(T) == 8) {
        if (c->force && contig) launch(lbm::lbm_two_steps<T, KIND, ARITH, true, true>);
        else if (c->force) launch(lbm::lbm_two_steps<T, KIND, ARITH, true, false>);
    }
    if (!c->force && contig) launch(lbm::lbm_two_steps<T, KIND, ARITH, false, true>);
    else if (!c->force) launch(lbm::lbm_two_steps<T, KIND, ARITH, false, false>);
    LBM_HIP_CHECK(hipGetLastError(), "two-step launch");
    return LBM_OK;
}

int launch_two_steps_opencl(StepPlan* c, const void* src, void* dst, int macro_last);  // lbm_two_step_opencl.hip

}  // namespace lbm_host
