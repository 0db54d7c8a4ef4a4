// lbm_two_step.hpp -- two collide-stream iterations in one pass over memory.
//
// A single step is bound by HBM (read and write every population once, 152 B
// per cell in FP32).  This kernel reads the lattice of iteration t and writes
// the one of iteration t + 2: the iteration in between lives in registers and
// LDS only, which halves the traffic per iteration.  Every value is computed by
// the same expressions as in the single-step kernels, so the results are
// theirs, bit for bit.
//
// A block owns a tile of columns (x, y), one per thread, and sweeps it along z
// over a chunk of planes.  The first iteration is computed on the whole tile,
// the second on the tile without its rim (except where the rim is the
// lattice's), so neighbouring tiles overlap by two columns and two rows.  Per
// plane p of the sweep a thread
//   1. has gathered the 19 populations of its cell in plane p (loads issued
//      one plane ahead), and issues those of plane p + 1;
//   2. collides them (first iteration) and exchanges the 16 populations that
//      move in x or y with its neighbours through LDS;
//   3. (output columns) collides the cell of plane p - 1 (second iteration):
//      the populations that move towards -z come from plane p, those that stay
//      in their plane were exchanged one plane ago, those that move towards +z
//      two planes ago -- both kept in registers.  The result is stored in the
//      next plane's round, before that round's loads, so that no wait for a
//      load ever waits for a store issued after it.
// One barrier per plane: the exchange buffer is double.
//
// Addresses: within a plane the slot of a cell relative to the plane's first
// slot, rel(c') = 19 c' - 18 (c' mod S) for S < N^2 and c' for S >= N^2, does
// not depend on z.  So a thread's source offsets are 32-bit registers set once,
// and a plane only needs the wavefront-uniform bases of its three source planes.
//
// Wall cells are in no tile.  The first iteration gathers from them in memory;
// what the second one takes from them is the same, their slots holding the
// initial lattice's values in both lattices (lbm_ctx::walls_initial): the
// initial population of the cell it arrives at -- the lid layer's equilibrium
// in the plane N - 2, w_i below it.
//
// What bounds it: on large lattices in FP32 memory, with arithmetic not far behind;
// at 128^3 and in FP64 a round's latency.  Measured at 512^3, FP32, stride 4096:
// 2.09 ms per iteration against 3.28 for the single step, the same without the
// arithmetic (2.0), 1.05 with the arithmetic alone; the VALU is busy 0.74 of the
// time.  A pair moves 2.10e10 bytes (1.04 times one read and one write of the
// lattice) at 5.0 TB/s, where the single step moves 6.2: the tile's rows are loaded
// by two blocks, which share them through L2.  128^3, stride 64: FP32 37 us an
// iteration at 4.8 TB/s with the VALU busy 0.59 of the time, FP64 69 us at 4.7 TB/s
// and 0.35 -- a plane's loads, LDS and barrier follow one another, and two
// wavefronts per SIMD (FP64) hide little of it.  Prefetching two planes instead of one gains nothing (2.07 without the
// arithmetic); tiles whose rows are not whole aligned 256-byte pieces lose most
// of the gain (3.4 ms).  FP64: 4.35 against 6.6 ms.
#pragma once

#include "lbm_kernels.hpp"

namespace lbm {

// Threads of a block: as many as a CU's registers hold with the state of one
// column each (19 populations in flight, 19 waiting for their plane, 19 at work:
// FP32 128 registers, FP64 256).
template <class T> struct TwoStepThreads {
    static constexpr int value = sizeof(T) == 4 ? 1024 : 512;
};

// LDS plane of population i of the exchange (those with e_x or e_y non-zero), else -1
__host__ __device__ constexpr int exchange_slot(int i) { return (i >= 7) ? i - 3 : (i >= 1 && i <= 4) ? i - 1 : -1; }

// A register value the compiler cannot see through: keeps a loop-invariant 32-bit
// offset from being widened outside the loop, where the (scalar base, 32-bit
// vector offset) form of the memory instructions is no longer recognised.
__device__ __forceinline__ void opaque(uint32_t& v) { asm volatile("" : "+v"(v)); }

// base (wavefront-uniform) + off bytes, in that form
template <class P, class E> __device__ __forceinline__ P* at_bytes(E* base, uint32_t off) {
    using B = typename std::conditional<std::is_const<E>::value, const char, char>::type;
    const uint64_t v = reinterpret_cast<uint64_t>(base);
    const uint64_t u = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v)))) |
                       (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32)))) << 32);
    return reinterpret_cast<P*>(reinterpret_cast<B*>(u) + off);
}

template <class T> struct TwoStepArgs {
    StepArgs<T> s;
    int32_t zlen;        // output planes per block
    int32_t tiles_x, tiles_y;
    int32_t w;           // columns of a tile's segment of a row (a power of two)
    int32_t rows;        // rows of a tile
    int32_t halo;        // the threads after the segments' have the columns beside them
    int32_t macro_last;  // store rho and u of the second iteration
};

// finish_type() without branches, for a non-wall column's flags plus its plane's
__device__ __forceinline__ int32_t interior_type(int32_t t) {
    const bool corner = ((t & (LEFT | RIGHT)) != 0) & ((t & (BOTTOM | TOP)) != 0) & ((t & BACK) != 0);
    return corner ? CORNER : (t == FRONT ? (FRONT | MOVING) : (t == NONE ? FLUID : t));
}

// collide_any() of a wavefront: without the boundary cases where it has none,
// and away from the lid (`lid`: the cells are in its plane) with the fluid's
// collision for all and a choice per population -- next to a side wall a
// wavefront holds a few bounce-back cells, and branches would cost it the
// registers of both sides.
template <class T, int ARITH>
__device__ __forceinline__ void collide_wave(int32_t t, bool lid, T (&f)[Q], T& rho, T& ux, T& uy, T& uz,
                                             const StepConsts<T>& k) {
    if (__builtin_amdgcn_ballot_w64(t != FLUID) == 0) {
        collide_any<T, ARITH>(FLUID, f, rho, ux, uy, uz, k);
    } else if (!lid) {
        constexpr int OPP[Q] = {0, 3, 4, 1, 2, 6, 5, 9, 10, 7, 8, 17, 18, 15, 16, 13, 14, 11, 12};
        T g[Q];
#pragma unroll
        for (int i = 0; i < Q; ++i) g[i] = f[i];
        collide_any<T, ARITH>(FLUID, g, rho, ux, uy, uz, k);
        const bool fluid = t == FLUID, back = is_bounceback(t);
#pragma unroll
        for (int i = 0; i < Q; ++i) g[i] = fluid ? g[i] : (back ? f[OPP[i]] : f[i]);
#pragma unroll
        for (int i = 0; i < Q; ++i) f[i] = g[i];
    } else {
        collide_any<T, ARITH>(t, f, rho, ux, uy, uz, k);
    }
}

// CONTIG: the cells of a row are contiguous (stride >= N)
template <class T, int KIND, int ARITH, bool FORCE, bool CONTIG>
__global__ __launch_bounds__((TwoStepThreads<T>::value)) void lbm_two_steps(TwoStepArgs<T> a) {
    using C = Codec<T, KIND>;
    using S = typename C::S;
    constexpr int THREADS = TwoStepThreads<T>::value;
    constexpr int PLANE = THREADS + 32;   // LDS elements of one exchanged population: at most 16 rows, two more columns each
    __shared__ S xch[2 * 16 * PLANE];
    __shared__ T force_of[FORCE ? 3 * THREADS : 1];  // body force at the threads' cells of the plane before
    __shared__ T lid_eq[Q];  // read next to walls only: from LDS, so that it does not occupy scalar registers
    const C codec{a.s.scale, a.s.inv_scale};
    const int32_t n = a.s.n;
    const int64_t n2 = int64_t(n) * n;

    const uint32_t lb = xcd_logical_block(blockIdx.x, gridDim.x, a.s.xcd_remap);
    const int32_t xt = int32_t(lb % uint32_t(a.tiles_x));
    const int32_t yt = int32_t((lb / uint32_t(a.tiles_x)) % uint32_t(a.tiles_y));
    const int32_t zc = int32_t(lb / uint32_t(a.tiles_x * a.tiles_y));
    const int32_t z0 = 1 + zc * a.zlen;
    const int32_t z1 = (z0 + a.zlen < n - 1) ? z0 + a.zlen : n - 1;  // output planes z0 .. z1 - 1
    const bool x_first = xt == 0, x_last = xt == a.tiles_x - 1;

    // Wall positions of the exchange are written by nobody: they hold what gathers
    // from wall cells supply, w_i but for the last planes (below).
    if (threadIdx.x < Q) lid_eq[threadIdx.x] = a.s.lid_eq[threadIdx.x];
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        if (exchange_slot(i) < 0) continue;
        const S rest = value_out<ARITH>(codec, (ARITH == AR_DELTA) ? T(0) : w_of<T>(i), w_of<T>(i));
        for (int k = int(threadIdx.x); k < PLANE; k += THREADS)
            xch[exchange_slot(i) * PLANE + k] = xch[(16 + exchange_slot(i)) * PLANE + k] = rest;
    }
    __syncthreads();

    // The thread's column: thread l of row r has column l of the tile's segment of
    // the row, so that its stores are whole aligned lines.  The columns on either
    // side of the segment are the halo threads', or else, of a row made of one or
    // two segments, that of the thread at the segment's other end, whose own is
    // the wall.  (Rows start at different wavefronts of their segment, so that
    // those with cells next to the wall spread over the SIMDs.)  Threads left over
    // repeat thread 0's loads.
    const int tid = int(threadIdx.x);
    const int h = tid - a.w * a.rows;
    const bool spare = h >= (a.halo ? 2 * a.rows : 0);
    const int r = spare ? 0 : (h < 0 ? tid / a.w : (h < a.rows ? h : h - a.rows));
    const int l = spare ? 0 : (h < 0 ? (tid + 64 * r) & (a.w - 1) : (h < a.rows ? -1 : a.w));
    const bool wall_lane = (x_first && l == 0) || (x_last && l == a.w - 1);
    const int col = (wall_lane && !a.halo && !(x_first && x_last)) ? (x_first ? a.w : -1) : l;
    const int32_t xc = xt * a.w + col, yc = yt * (a.rows - 2) + r;
    const bool in_tile = !spare && xc >= 1 && xc <= n - 2 && yc >= 1 && yc <= n - 2;
    const bool out = in_tile && h < 0 && !wall_lane && r >= 1 && r <= a.rows - 2;
    const int32_t x = min(max(xc, 1), n - 2), y = min(max(yc, 1), n - 2);

    const int64_t smask = a.s.stride - 1;
    const uint32_t pmask = uint32_t(a.s.stride < n2 ? smask : n2 - 1);
    auto rel = [&](int32_t xx, int32_t yy) -> uint32_t {  // bytes from the plane's first slot
        const uint32_t c = uint32_t(xx + n * yy);
        return (a.s.stride < n2 ? 19u * c - 18u * (c & pmask) : c) * uint32_t(sizeof(S));
    };
    uint32_t off[3][3];  // [e_y + 1][e_x + 1]: source column of a gather (CONTIG: e_x = 0 only)
#pragma unroll
    for (int ey = -1; ey <= 1; ++ey)
#pragma unroll
        for (int ex = -1; ex <= 1; ++ex) off[ey + 1][ex + 1] = rel(x - ex, y - ey);
    uint32_t& own = off[1][1];
    auto plane = [&](int32_t z) __attribute__((always_inline)) -> int64_t {  // slot of the plane's first cell, population 0
        const int64_t c = n2 * z;
        return 19 * c - 18 * (c & smask);
    };

    const S* __restrict__ src = static_cast<const S*>(a.s.src);
    S* __restrict__ dst = static_cast<S*>(a.s.dst);
    S L[Q];
    T G[3] = {T(0), T(0), T(0)};  // body force at the cell, with the same plane's populations
    auto issue = [&](int32_t p) __attribute__((always_inline)) {
        if (p == 0 || p == n - 1) return;  // a wall plane
        const int64_t b[3] = {plane(p + 1), plane(p), plane(p - 1)};
#pragma unroll
        for (int k = 0; k < 9; ++k)
            if (!CONTIG || k % 3 == 1) opaque(off[k / 3][k % 3]);
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            const S* base = src + (b[ez_of(i) + 1] + int64_t(i) * a.s.stride);
            if constexpr (CONTIG) L[i] = *(at_bytes<const S>(base, off[ey_of(i) + 1][1]) - ex_of(i));
            else L[i] = *at_bytes<const S>(base, off[ey_of(i) + 1][ex_of(i) + 1]);
        }
        if constexpr (FORCE) {
            uint32_t cell = uint32_t(x + n * y) * uint32_t(sizeof(T));
            opaque(cell);
#pragma unroll
            for (int d = 0; d < 3; ++d) G[d] = *at_bytes<const T>(a.s.force + (int64_t(d) * a.s.n3 + n2 * p), cell);
        }
    };
    auto store = [&](const S (&o)[Q], int32_t z) __attribute__((always_inline)) {
        const int64_t b = plane(z);
        opaque(own);
#pragma unroll
        for (int i = 0; i < Q; ++i) LBM_LAT_STORE(o[i], at_bytes<S>(dst + (b + int64_t(i) * a.s.stride), own));
    };
    // what the gather of population i from a wall cell of plane z supplies
    auto wall_value = [&](int i, int32_t z) __attribute__((always_inline)) -> S {
        const T rest = (ARITH == AR_DELTA) ? T(0) : w_of<T>(i);
        return value_out<ARITH>(codec, z + ez_of(i) == n - 2 ? lid_eq[i] : rest, w_of<T>(i));
    };
    const int32_t xf = x_flags(x, n) | row_flags(y, 2, n);  // flags of the column in a plane away from the z walls
    const int32_t t_mid = interior_type(xf);
    auto column_type = [&](int32_t z) __attribute__((always_inline)) -> int32_t {  // of an interior plane
        return (z == 1 || z == n - 2) ? interior_type(xf | (z == 1 ? BACK : 0) | (z == n - 2 ? FRONT : 0)) : t_mid;
    };
    S A0[Q];  // populations with e_z = 0, gathered one plane ago (elements of the others unused)
    S B1[Q];  // e_z = +1, gathered one plane ago
    S B2[Q];  // e_z = +1, gathered two planes ago
    S o[Q];   // the second iteration's result, stored in the next round
    const int pitch = a.w + 2;
    const int lds_own = r * pitch + col + 1;  // position of column (xt w + c, yt (rows - 2) + r): r pitch + c + 1

    issue(z0 - 1);
    for (int32_t p = z0 - 1; p <= z1; ++p) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this plane's loads (and the stores of a round ago)
        S v[Q];
#pragma unroll
        for (int i = 0; i < Q; ++i) v[i] = L[i];
        if (out && p - 2 >= z0) store(o, p - 2);
        T F0[3], F1[3];  // body force at the cells of planes p - 1 and p
        if constexpr (FORCE) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                F0[d] = force_of[d * THREADS + tid];
                F1[d] = G[d];
                force_of[d * THREADS + tid] = G[d];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (p < z1) issue(p + 1);
        __builtin_amdgcn_sched_barrier(0);
        T rho, ux, uy, uz;
        if (p == 0 || p == n - 1) {
#pragma unroll
            for (int i = 0; i < Q; ++i) v[i] = wall_value(i, p);
        } else {
            const int32_t t = column_type(p);
            T f[Q];
#pragma unroll
            for (int i = 0; i < Q; ++i) f[i] = value_in<ARITH>(codec, v[i], w_of<T>(i));
            collide_wave<T, ARITH>(t, p == n - 2, f, rho, ux, uy, uz, a.s.k);
            if constexpr (FORCE) add_force_any<T, ARITH>(t, f, F1[0], F1[1], F1[2], a.s.k);
#pragma unroll
            for (int i = 0; i < Q; ++i) v[i] = value_out<ARITH>(codec, f[i], w_of<T>(i));
        }
        S* const x_own = xch + ((p & 1) * 16 * PLANE + lds_own);
        if (in_tile) {
#pragma unroll
            for (int i = 0; i < Q; ++i)
                if (exchange_slot(i) >= 0) x_own[exchange_slot(i) * PLANE] = v[i];
        }
        if (p >= n - 3) {  // gathers that arrive in the plane below the lid
            for (int k = tid; k < a.rows * pitch; k += THREADS) {
                const int32_t xw = xt * a.w + k % pitch - 1, yw = yt * (a.rows - 2) + k / pitch;
                if (xw == 0 || xw == n - 1 || yw == 0 || yw == n - 1) {
#pragma unroll
                    for (int i = 0; i < Q; ++i)
                        if (exchange_slot(i) >= 0 && p + ez_of(i) == n - 2)
                            xch[((p & 1) * 16 + exchange_slot(i)) * PLANE + k] = wall_value(i, p);
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (out) {
            const S* const x_row[3] = {x_own + pitch, x_own, x_own - pitch};  // [e_y + 1]: the row it comes from
            // population i of the first iteration, arriving at this column in plane p + e_z
            auto arriving = [&](int i) __attribute__((always_inline)) -> S {
                if (exchange_slot(i) < 0) return v[i];
                return x_row[ey_of(i) + 1][exchange_slot(i) * PLANE - ex_of(i)];
            };
            if (p >= z0 + 1) {
                const int32_t z = p - 1;
                T g[Q];
#pragma unroll
                for (int i = 0; i < Q; ++i)
                    g[i] = value_in<ARITH>(codec, ez_of(i) < 0 ? arriving(i) : (ez_of(i) == 0 ? A0[i] : B2[i]), w_of<T>(i));
                const int32_t t = column_type(z);
                collide_wave<T, ARITH>(t, z == n - 2, g, rho, ux, uy, uz, a.s.k);
                if constexpr (FORCE) add_force_any<T, ARITH>(t, g, F0[0], F0[1], F0[2], a.s.k);
                if (a.macro_last && is_store_macro(t)) {
                    uint32_t cell = uint32_t(x + n * y) * uint32_t(sizeof(T));
                    opaque(cell);
                    *at_bytes<T>(a.s.rho + n2 * z, cell) = rho;
                    *at_bytes<T>(a.s.u + n2 * z, cell) = ux;
                    *at_bytes<T>(a.s.u + (a.s.n3 + n2 * z), cell) = uy;
                    *at_bytes<T>(a.s.u + (2 * a.s.n3 + n2 * z), cell) = uz;
                }
#pragma unroll
                for (int i = 0; i < Q; ++i) o[i] = value_out<ARITH>(codec, g[i], w_of<T>(i));
            }
#pragma unroll
            for (int i = 0; i < Q; ++i) {
                if (ez_of(i) == 0) A0[i] = arriving(i);
                if (ez_of(i) > 0) {
                    B2[i] = B1[i];
                    B1[i] = arriving(i);
                }
            }
        }
    }
    if (out) store(o, z1 - 1);
}

}  // namespace lbm
