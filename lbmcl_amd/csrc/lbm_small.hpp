// lbm_small.hpp -- several collide-stream iterations of a small lattice in one
// launch.
//
// Up to 32^3 an iteration takes little longer than the launch that does it.  Here a block takes k iterations of a tile of
// cells: it computes the first one on the tile widened by k - 1 cells on every
// side, the next on a region one cell smaller, and so on down to the tile
// itself, with the populations in LDS in between.  Nothing waits for another
// block; what neighbouring tiles have in common is computed by both.  A lattice
// that is one tile (8^3) needs no widening, and takes any number of iterations
// in one launch.
//
// The first iteration gathers from memory, the last one stores to memory, those
// in between are in place: every thread gathers its cells' populations and
// collides them, a barrier, then it writes them back.  Every value is computed
// by the single-step kernels' expressions and rounded to the stored type after
// each iteration, so the results are theirs, bit for bit.
//
// Wall cells next to the region are in LDS too, with what gathers from them
// supply: their slots hold the initial lattice's values in both lattices
// (lbm_ctx::walls_initial), the lid layer's equilibrium or w_i.
//
// What bounds it: the instructions of one wavefront after another.  An 8^3
// iteration is 216 cells, one wavefront per SIMD at most, and takes 1.0 us in
// FP32 (1.4 in FP64), against 3.7 for a launch; three iterations of 32^3 take 9.9
// us, of which the launch is about 3.
#pragma once

#include "lbm_two_step.hpp"

namespace lbm {

// A tile of X x Y x Z cells, widened by G on every side: the box in LDS.
template <int X_, int Y_, int Z_, int G_> struct SmallTile {
    static constexpr int X = X_, Y = Y_, Z = Z_, G = G_;
    static constexpr int W = X + 2 * G, H = Y + 2 * G, CELLS = W * H * (Z + 2 * G);
    static constexpr int THREADS = (CELLS + 63) / 64 * 64;  // a cell a thread in the first iteration
    static_assert(THREADS <= 1024, "one cell per thread");
};

template <class T> struct SmallArgs {
    StepArgs<T> s;         // s.dst: the lattice of the last iteration
    void* prev;            // a lattice of one tile: the lattice of the last but one, else null
    int32_t tiles_x, tiles_y;
    int32_t k;             // iterations: at most G + 1, or any number of a lattice of one tile
    int64_t every, phase;  // rho and u are stored by iterations j = 1 .. k with (phase + j) % every == 0 (every > 0)
};

// The collision of any interior cell without branches between its kinds: what
// collide_any() computes for the lane's own kind, chosen population by
// population.  In a small lattice most wavefronts hold several kinds, and a
// branch for each costs the sum of their instructions.
template <class T, int ARITH>
__device__ __forceinline__ void collide_blend(int32_t t, T (&f)[Q], T& rho, T& ux, T& uy, T& uz, const StepConsts<T>& k) {
    constexpr int PI[9] = {1, 2, 6, 7, 10, 15, 16, 11, 12};  // e_i
    constexpr int PO[9] = {3, 4, 5, 9, 8, 13, 14, 17, 18};   // -e_i
    const bool moving = is_moving(t), back = is_bounceback(t), keeps = !moving && t != FLUID;
    f[5] = moving ? f[6] : f[5];  // the lid fix-up of moments()
    f[11] = moving ? f[17] : f[11];
    f[12] = moving ? f[18] : f[12];
    f[13] = moving ? f[15] : f[13];
    f[14] = moving ? f[16] : f[14];
    T g[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) g[i] = f[i];
    if constexpr (ARITH == AR_EXACT || ARITH == AR_OPENCL) {
        const int32_t fluid = FLUID;
        moments<T>(fluid, g, rho, ux, uy, uz, k);
        ux = moving ? k.U : ux;
        uy = moving ? T(0) : uy;
        uz = moving ? T(0) : uz;
        const T u2 = (ARITH == AR_OPENCL) ? u2_contracted<T>(ux, uy, uz) : ((ux * ux) + (uy * uy)) + (uz * uz);
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            if constexpr (ARITH == AR_OPENCL) {
                const T e = feq_contracted<T>(i, rho, ux, uy, uz, u2);
                g[i] = moving ? e : fma_any<T>(k.inv_tau, e - f[i], f[i]);
            } else {
                const T e = feq<T>(i, rho, ux, uy, uz, u2);
                g[i] = moving ? e : f[i] + k.inv_tau * (e - f[i]);
            }
        }
    } else {
        collide_any<T, ARITH>(FLUID, g, rho, ux, uy, uz, k);
        if (__builtin_amdgcn_ballot_w64(moving) != 0) {
            T m[Q], mr, mx, my, mz;
#pragma unroll
            for (int i = 0; i < Q; ++i) m[i] = f[i];
            collide_any<T, ARITH>(FRONT | MOVING, m, mr, mx, my, mz, k);
#pragma unroll
            for (int i = 0; i < Q; ++i) g[i] = moving ? m[i] : g[i];
            rho = moving ? mr : rho;
            ux = moving ? mx : ux;
            uy = moving ? my : uy;
            uz = moving ? mz : uz;
        }
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const T a = f[PI[q]], b = f[PO[q]];
        f[PI[q]] = keeps ? (back ? b : a) : g[PI[q]];
        f[PO[q]] = keeps ? (back ? a : b) : g[PO[q]];
    }
    f[0] = keeps ? f[0] : g[0];
}

template <class T, int KIND, int ARITH, class TILE>
__global__ __launch_bounds__((TILE::THREADS)) void lbm_small_steps(SmallArgs<T> a) {
    using C = Codec<T, KIND>;
    using S = typename C::S;
    constexpr int W = TILE::W, H = TILE::H, G = TILE::G, CELLS = TILE::CELLS;
    __shared__ S pop[Q * CELLS];
    const C codec{a.s.scale, a.s.inv_scale};
    const int32_t n = a.s.n, k = a.k;
    const int tid = int(threadIdx.x);

    const uint32_t lb = xcd_logical_block(blockIdx.x, gridDim.x, a.s.xcd_remap);
    const int32_t lo[3] = {1 + int32_t(lb % uint32_t(a.tiles_x)) * TILE::X,
                           1 + int32_t((lb / uint32_t(a.tiles_x)) % uint32_t(a.tiles_y)) * TILE::Y,
                           1 + int32_t(lb / uint32_t(a.tiles_x * a.tiles_y)) * TILE::Z};
    const int32_t hi[3] = {min(lo[0] + TILE::X, n - 1), min(lo[1] + TILE::Y, n - 1), min(lo[2] + TILE::Z, n - 1)};  // past the tile

    const S* const src = static_cast<const S*>(a.s.src);
    const uint32_t smask = uint32_t(a.s.stride - 1), stride = uint32_t(a.s.stride);
    // slot of (cell c, population i), 32 bits (n <= 32)
    auto slot32 = [&](uint32_t c, int i) __attribute__((always_inline)) -> uint32_t {
        return 19u * c - 18u * (c & smask) + uint32_t(i) * stride;
    };

    {  // walls of the box: position tid
        const int32_t x = lo[0] - G + tid % W, y = lo[1] - G + (tid / W) % H, z = lo[2] - G + tid / (W * H);
        if (tid < CELLS && (x == 0 || y == 0 || z == 0 || x == n - 1 || y == n - 1 || z == n - 1)) {
#pragma unroll
            for (int i = 0; i < Q; ++i) {
                const T rest = (ARITH == AR_DELTA) ? T(0) : w_of<T>(i);
                pop[i * CELLS + tid] = value_out<ARITH>(codec, z + ez_of(i) == n - 2 ? a.s.lid_eq[i] : rest, w_of<T>(i));
            }
        }
    }

    int64_t phase = a.phase;
    int region = -1;  // widening the cell below was placed in
    int at = -1;      // its position in the box; negative: none
    uint32_t c = 0;
    int32_t t = FLUID;
    bool own = false;
    for (int32_t s = 1; s <= k; ++s) {
        bool macro = false;
        if (a.every > 0) {
            phase = phase + 1 == a.every ? 0 : phase + 1;
            macro = phase == 0;
        }
        const int32_t g = min(k - s, G);  // the region: the tile widened by g, inside the walls
        if (g != region && (region < 0 || a.prev == nullptr)) {  // the same cells throughout in a lattice of one tile
            region = g;
            const int32_t r0[3] = {max(lo[0] - g, 1), max(lo[1] - g, 1), max(lo[2] - g, 1)};
            const int32_t rw = min(hi[0] + g, n - 1) - r0[0], rh = min(hi[1] + g, n - 1) - r0[1],
                          rd = min(hi[2] + g, n - 1) - r0[2];
            // quotients by float: exact below 2^16
            const int row = int((float(tid) + 0.5f) * (1.0f / float(rw)));
            const int zz = int((float(row) + 0.5f) * (1.0f / float(rh)));
            const int32_t x = r0[0] + tid - row * rw, y = r0[1] + row - zz * rh, z = r0[2] + zz;
            c = uint32_t(x + n * (y + n * z));
            at = tid < rw * rh * rd ? (x - lo[0] + G) + W * ((y - lo[1] + G) + H * (z - lo[2] + G)) : -1;
            t = interior_type(x_flags(x, n) | row_flags(y, z, n));
            own = x >= lo[0] && x < hi[0] && y >= lo[1] && y < hi[1] && z >= lo[2] && z < hi[2];
        }
        const bool first = s == 1, last = s == k;
        T f[Q];
        T F[3] = {T(0), T(0), T(0)};  // body force, loaded with the populations
        if (at >= 0) {
            if (a.s.force) {
#pragma unroll
                for (int d = 0; d < 3; ++d) F[d] = a.s.force[int64_t(d) * a.s.n3 + c];
            }
            if (first) {
                S h[Q];
#pragma unroll
                for (int i = 0; i < Q; ++i)
                    h[i] = src[slot32(c - uint32_t(ex_of(i) + n * (ey_of(i) + n * ez_of(i))), i)];
#pragma unroll
                for (int i = 0; i < Q; ++i) f[i] = value_in<ARITH>(codec, h[i], w_of<T>(i));
            } else {
                const S* const p = pop + at;
#pragma unroll
                for (int i = 0; i < Q; ++i)
                    f[i] = value_in<ARITH>(codec, p[i * CELLS - (ex_of(i) + W * (ey_of(i) + H * ez_of(i)))], w_of<T>(i));
            }
        }
        // everyone has gathered (in the first iteration: has read the source lattice, which `prev` may be)
        if (!last || a.prev) __syncthreads();
        if (at >= 0) {
            T rho, ux, uy, uz;
            if (__builtin_amdgcn_ballot_w64(t != FLUID) == 0) collide_any<T, ARITH>(FLUID, f, rho, ux, uy, uz, a.s.k);
            else collide_blend<T, ARITH>(t, f, rho, ux, uy, uz, a.s.k);
            if (a.s.force) add_force_any<T, ARITH>(t, f, F[0], F[1], F[2], a.s.k);
            if (macro && own && is_store_macro(t)) {
                a.s.rho[c] = rho;
                a.s.u[c] = ux;
                a.s.u[a.s.n3 + c] = uy;
                a.s.u[2 * a.s.n3 + c] = uz;
            }
            if (!last) {
                S* const p = pop + at;
#pragma unroll
                for (int i = 0; i < Q; ++i) p[i * CELLS] = value_out<ARITH>(codec, f[i], w_of<T>(i));
            }
            if (last || (a.prev && s == k - 1)) {
                S* const dst = static_cast<S*>(last ? a.s.dst : a.prev);
#pragma unroll
                for (int i = 0; i < Q; ++i) dst[slot32(c, i)] = value_out<ARITH>(codec, f[i], w_of<T>(i));
            }
        }
        if (!last) __syncthreads();  // this iteration's values are in place
    }
}

}  // namespace lbm
