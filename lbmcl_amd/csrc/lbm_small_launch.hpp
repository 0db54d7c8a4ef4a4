// lbm_small_launch.hpp -- launching the small-lattice kernel, shared by the two
// translation units that instantiate it.
#pragma once

#include "lbm_ctx.hpp"
#include "lbm_small.hpp"

namespace lbm_host {

// Tiles, the fastest of those tried (us per iteration; single steps / 4 x 4 x 4
// widened by 1, 2, 3 / 8 x 4 x 4 by 1, 2 / 8 x 8 x 8 by 1): 16^3 FP32 4.3 / 3.2, 2.7,
// 2.9 / 3.4, 3.0 / 4.2; 32^3 FP32 4.7 / 3.8, 3.8, 5.6 / 3.6, 3.3 / 5.1, FP64 5.0 / 4.5,
// 5.6, 6.9 / 4.2, 4.2 / 5.9.  Wider regions take fewer launches but compute more
// cells twice.  At 64^3 the chip has no idle CUs left for those (FP32 8.4 / 12.8,
// 15.6, 38 / 10.7, 13.5 / 9.7, FP64 with a force 13.3 / 15.3 at best, FP16 7.7 / 11.2
// at best): single steps.  8^3: FP32 3.7 / 1.0, FP64 3.9 / 1.4.
using SmallTile8 = lbm::SmallTile<6, 6, 6, 1>;
using SmallTile16 = lbm::SmallTile<4, 4, 4, 2>;
using SmallTile32 = lbm::SmallTile<8, 4, 4, 2>;

template <class T, int KIND, int ARITH, class TILE>
inline int launch_small_tile(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase) {
    lbm::SmallArgs<T> a{};
    a.s = step_args<T, ARITH>(c, src, dst, 0, 0);
    a.prev = prev;
    a.k = k;
    a.every = every;
    a.phase = phase;
    const int32_t w = c->n - 2;
    a.tiles_x = (w + TILE::X - 1) / TILE::X;
    a.tiles_y = (w + TILE::Y - 1) / TILE::Y;
    const int32_t tiles_z = (w + TILE::Z - 1) / TILE::Z;
    launch_on(c, lbm::lbm_small_steps<T, KIND, ARITH, TILE>, dim3(unsigned(a.tiles_x * a.tiles_y * tiles_z)),
              dim3(TILE::THREADS), nullptr, nullptr, a);
    LBM_HIP_CHECK(hipGetLastError(), "small-lattice launch");
    return LBM_OK;
}

template <class T, int KIND, int ARITH>
inline int launch_small_impl(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase) {
    if (c->n <= 8) return launch_small_tile<T, KIND, ARITH, SmallTile8>(c, src, dst, prev, k, every, phase);
    if (c->n == 16) return launch_small_tile<T, KIND, ARITH, SmallTile16>(c, src, dst, prev, k, every, phase);
    return launch_small_tile<T, KIND, ARITH, SmallTile32>(c, src, dst, prev, k, every, phase);
}

int launch_small_opencl(StepPlan* c, const void* src, void* dst, void* prev, int32_t k, int64_t every, int64_t phase);

}  // namespace lbm_host
