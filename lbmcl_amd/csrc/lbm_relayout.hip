// lbm_relayout.hip -- long ranges of iterations on lattices with short runs: the
// lattice is put into the layout that the kernels read fastest, iterated there,
// and put back.
//
// With a CSoA stride of less than 128 bytes a line holds several populations of
// the same cells.  The kernels then fetch lines that they use in part (or, the
// tile kernel, move everything through LDS twice), and two iterations in one
// launch cost more than two launches.  Measured, us per iteration at the stride
// given / at 4096:
//   FP32   128^3 stride 1 73 / 35, 8 64 / 35, 16 45 / 35, 32 37 / 35; 256^3 stride 1
//          557 / 264, 16 373 / 264, 32 275 / 264; 64^3 stride 1 12.4 / 8.4
//   FP64   128^3 stride 1 147 / 68, 4 113 / 68, 8 79 / 68, 16 70 / 68
//   FP16   128^3 stride 1 48.5 / 29.0, 32 49.5 / 29.0; 256^3 stride 32 294 / 217
// Changing the layout reads and writes a lattice once; a range needs it three
// times (the source, and the last two states): 200 us at 128^3 FP32 and 1.8 ms at
// 256^3, as long as six or seven iterations there.
#include "lbm_range.hpp"

namespace {

constexpr int kCells = 256;  // cells of a block, one per thread

// The stored values of kCells consecutive cells, in one piece in the layout with
// the smaller stride (at most kCells), and in a run per population in the other
// (a multiple of kCells).  Through LDS, so that both sides are whole lines.
// `small_in`: the smaller stride is the source's.
//
// What bounds it: memory.
template <class U, bool SMALL_IN>
__global__ __launch_bounds__(kCells) void relayout_kernel(const U* in, U* out, int32_t log2_small, int64_t large) {
    __shared__ U v[lbm::Q * kCells];
    const int t = int(threadIdx.x);
    const int64_t c0 = int64_t(blockIdx.x) * kCells;
    const int64_t piece = 19 * c0, run = 19 * c0 - 18 * (c0 & (large - 1)) + t;
    const int at = (((t >> log2_small) * lbm::Q) << log2_small) + (t & ((1 << log2_small) - 1));
    if constexpr (SMALL_IN) {
#pragma unroll
        for (int i = 0; i < lbm::Q; ++i) v[i * kCells + t] = __builtin_nontemporal_load(in + piece + i * kCells + t);
    } else {
#pragma unroll
        for (int i = 0; i < lbm::Q; ++i) v[at + (i << log2_small)] = __builtin_nontemporal_load(in + run + i * large);
    }
    __syncthreads();
    if constexpr (SMALL_IN) {
#pragma unroll
        for (int i = 0; i < lbm::Q; ++i) out[run + i * large] = v[at + (i << log2_small)];
    } else {
#pragma unroll
        for (int i = 0; i < lbm::Q; ++i) out[piece + i * kCells + t] = v[i * kCells + t];
    }
}

}  // namespace

namespace lbm_host {

// From 64^3 on: smaller lattices have their own kernel and are read through the
// caches whole.
bool relayout_possible(const StepPlan* c) {
    return c->cfg.kernel == LBM_KERNEL_AUTO && c->n >= 64 && c->stride * int64_t(c->ssize) < 128;
}

// Where the three changes have paid for themselves: the fixed cost of a relaid range
// over what an iteration gains, the worst of storing rho and u never, every second
// and every iteration, with and without a force (which decide whether two steps go
// in one launch in either layout).  Measured, iterations at 64^3 / 128^3 / 256^3 / 512^3:
//   runs of at most 32 bytes    FP32 11 / 9 / 9 / 10, FP64 7 / 12 / 10, 16-bit 20 / 5 / 7
//   runs of 64 bytes            FP32 8 / 20 / 29 / 15, FP64 60 / 56 / 45 / 77, 16-bit 15 / 5 / 11 / 9
// (64^3 16-bit gains 2 us an iteration for 30, 64^3 FP64 with runs of 64 bytes 1 for
// 50, 128^3 11 for 450, 512^3 370 for 28000.)
bool relayout_pays(const StepPlan* c, int64_t count) {
    if (!relayout_possible(c)) return false;
    if (c->stride * int64_t(c->ssize) <= 32) return count >= (c->ssize == 2 && c->n == 64 ? 24 : 12);
    return count >= (c->ssize == 8 ? 96 : 32);
}

int relayout(lbm_ctx* c, const void* in, int64_t stride_in, void* out, int64_t stride_out) {
    const bool small_in = stride_in < stride_out;
    const int64_t small = std::min(stride_in, stride_out), large = std::max(stride_in, stride_out);
    if (small > kCells || large < kCells || c->n3 % kCells)
        return fail(LBM_ERR_INVALID, "no change of layout between these strides");
    const auto launch = [&](auto one) {
        using U = decltype(one);
        const dim3 grid{unsigned(c->n3 / kCells)};
        if (small_in)
            hipLaunchKernelGGL((relayout_kernel<U, true>), grid, dim3(kCells), 0, c->stream, static_cast<const U*>(in),
                               static_cast<U*>(out), ilog2(small), large);
        else
            hipLaunchKernelGGL((relayout_kernel<U, false>), grid, dim3(kCells), 0, c->stream, static_cast<const U*>(in),
                               static_cast<U*>(out), ilog2(small), large);
    };
    if (c->ssize == 8) launch(uint64_t());
    else if (c->ssize == 4) launch(uint32_t());
    else launch(uint16_t());
    LBM_HIP_CHECK(hipGetLastError(), "relayout launch");
    return LBM_OK;
}

}  // namespace lbm_host
