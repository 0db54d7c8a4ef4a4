// lbm_adjoint.hip -- gradients of a final-state objective with respect to the
// lid velocity U, the viscosity nu and a per-cell body force g(x), by the
// adjoint (reverse) collide-stream step with checkpointing.
//
// Schedule for T steps with checkpoints every K steps (M = ceil(T / K)
// segments):
//   forward   P_0 -> P_T; P_{mK} is kept for every segment m; the states of
//             the last segments are kept whole (their tapes), as many as memory
//             is plentiful for, so they need no recomputation.
//   seed      lambda_T = dJ/dP_T from the objective on the gathered P_T.
//   reverse   for m = M-1 .. 0: recompute P_{mK+1} .. P_{mK+len-1} from the
//             checkpoint into a tape (not where it is kept), then step
//             lambda backwards through the segment.
// Device memory: M checkpoints + (K - 1) states of a tape + 2 lattices + 2 adjoint
// lattices, i.e. about 2 sqrt(T) states for K = sqrt(T); and where K is not the
// caller's, the tapes that memory is plentiful for (lbm_tapes.hpp).
// No counterpart in the reference.
#include <type_traits>

#include "lbm_adjoint.hpp"
#include "lbm_range.hpp"
#include "lbm_tapes.hpp"

using namespace lbm_host;

namespace {

// How a gradient's steps run: its states, which nobody else sees, are in the
// fastest layout where the context's has short runs, and are each written once.
struct AdjointPlan {
    lbm_ctx* c;
    const int64_t own;
    explicit AdjointPlan(lbm_ctx* ctx) : c(ctx), own(ctx->stride) {
        c->alternates = false;
        if (relayout_possible(c)) c->stride = kFastStride;
    }
    ~AdjointPlan() {
        c->stride = own;
        c->alternates = true;
    }
};

// Device memory of one gradient, back in the pool at its end (allocate_gradient's
// allocator).
struct AdjointBuffers {
    lbm_ctx* c;
    std::vector<std::pair<void*, size_t>> owned;
    size_t free_bytes = 0, total_bytes = 0;
    explicit AdjointBuffers(lbm_ctx* ctx) : c(ctx) {}
    ~AdjointBuffers() {
        (void)hipStreamSynchronize(c->stream);  // an error may have left work enqueued
        for (const auto& b : owned) g_pool.give(c->cfg.device, b.first, b.second);
        g_pool.leave_half(c->cfg.device);
    }
    int alloc(void** p, size_t bytes, const char* what) {
        const int rc = pool_alloc(c, p, bytes, what);
        if (!rc) owned.emplace_back(*p, bytes);
        return rc;
    }
    bool try_alloc(void** p, size_t bytes) {
        const std::string last_error = g_last_error;
        if (!alloc(p, bytes, "adjoint tape")) return true;
        g_last_error = last_error;
        return false;
    }
    void give_back(size_t n) {  // to the device: memory is short
        for (; n > 0; --n, owned.pop_back()) (void)hipFree(owned.back().first);
    }
    size_t available() {
        if (hipMemGetInfo(&free_bytes, &total_bytes) != hipSuccess) {
            (void)hipGetLastError();
            free_bytes = total_bytes = 0;
            return 0;
        }
        return free_bytes + g_pool.held(c->cfg.device);
    }
    size_t total() const { return total_bytes; }  // as of the last available()
};

// Cells per lane of the vector adjoint kernel, 0 if it cannot run: it needs
// whole wavefronts per row (N / V >= 64), at most 512 threads per row, and V
// consecutive cells contiguous (stride >= V).  8-byte lanes where possible
// (FP32: V = 2), else one cell per lane.  LBM_KERNEL_GENERIC and
// LBM_KERNEL_ROW select the generic adjoint kernel.
template <class T> int64_t adjoint_vec_width(const lbm_ctx* c) {
    if (c->cfg.kernel == LBM_KERNEL_GENERIC || c->cfg.kernel == LBM_KERNEL_ROW) return 0;
    for (int64_t V : {int64_t(8 / sizeof(T)), int64_t(1)})
        if (c->n / V >= 64 && c->n / V <= 512 && c->stride >= V) return V;
    return 0;
}

template <class T>
int run_adjoint(lbm_ctx* c, const lbm_adjoint_config& cfg, lbm_adjoint_result* res, double* grad_g_host) {
    const int64_t T_steps = cfg.steps;
    int64_t K = cfg.checkpoint_every;
    if (K <= 0) K = int64_t(std::llround(std::sqrt(double(T_steps))));
    if (K < 1) K = 1;
    if (K > T_steps) K = T_steps;
    const int64_t M = (T_steps + K - 1) / K;
    const size_t S = size_t(c->n3) * lbm::Q * sizeof(T);
    AdjointPlan plan(c);
    AdjointBuffers buf(c);
    constexpr bool staged = std::is_same<T, float>::value;
    // vector adjoint kernel: one block of N / V threads per interior row
    const int64_t V = adjoint_vec_width<T>(c);
    const bool vec = V > 0;
    const int block = vec ? int(c->n / V) : 256;
    const int64_t nblocks = vec ? int64_t(c->n - 2) * (c->n - 2) : (c->n3 + 255) / 256;

    GradientSizes z;
    z.segments = M;
    z.tape = K - 1;
    z.state = S;
    // dJ/dg: FP64 sum; FP32 runs accumulate in an FP32 buffer flushed into it
    // every ADJ_FLUSH steps (half the read-modify-write traffic per step)
    z.grad = grad_g_host ? size_t(3 * c->n3) * sizeof(double) : 0;
    z.grad_stage = grad_g_host && staged ? size_t(3 * c->n3) * sizeof(T) : 0;
    z.partials = size_t(3 * nblocks) * sizeof(double);
    z.sums = 3 * sizeof(double);
    z.extra = cfg.checkpoint_every <= 0;
    const size_t memory = g_pool.device_memory();
    if (memory > 0 && needed_bytes(z) > double(memory))
        return fail(LBM_ERR_MEMORY, "a gradient of " + std::to_string(T_steps) + " steps with a checkpoint every " +
                                        std::to_string(K) + " needs " + std::to_string(needed_bytes(z) / 1e9) +
                                        " GB, more than the device has");
    GradientMemory mem;
    int rc = allocate_gradient(buf, z, &mem);
    if (rc) return rc;
    const double device_bytes = double(S) * double(2 + mem.checkpoints.size() + mem.tapes.size() + 2) + double(z.grad) +
                                double(z.grad_stage) + double(c->n3) * (4 * sizeof(T) + 4);

    // states: ckpt[0] is the context's lattice 0, the final state goes to lattice 1
    std::vector<void*> ckpt(1, c->lat[0]);
    ckpt.insert(ckpt.end(), mem.checkpoints.begin(), mem.checkpoints.end());
    // tapes: that of the last segment, which earlier ones recompute their states
    // into, and one more for each of the `kept` - 1 segments before it
    std::vector<void*>& tapes = mem.tapes;
    const auto is_kept = [&](int64_t m) { return m >= M - mem.kept; };
    const auto tape_of = [&](int64_t m) { return tapes.data() + (is_kept(m) ? M - 1 - m : 0) * z.tape; };
    void* const* const lam = mem.lambda;
    double* const grad_g = static_cast<double*>(mem.grad);
    T* const grad_acc = static_cast<T*>(staged ? mem.grad_stage : mem.grad);
    double* const partials = static_cast<double*>(mem.partials);
    double* const acc = static_cast<double*>(mem.sums);
    if (grad_g) LBM_HIP_CHECK(hipMemsetAsync(grad_g, 0, z.grad, c->stream), "hipMemsetAsync");
    if (grad_acc && staged) LBM_HIP_CHECK(hipMemsetAsync(grad_acc, 0, z.grad_stage, c->stream), "hipMemsetAsync");
    LBM_HIP_CHECK(hipMemsetAsync(partials, 0, z.partials, c->stream), "hipMemsetAsync");
    LBM_HIP_CHECK(hipMemsetAsync(acc, 0, z.sums, c->stream), "hipMemsetAsync");
    // slots that no step writes (fed by wall cells) must read as zero
    for (int j = 0; j < 2; ++j) LBM_HIP_CHECK(hipMemsetAsync(lam[j], 0, S, c->stream), "hipMemsetAsync");

    hipEvent_t e0, e1, e2;
    LBM_HIP_CHECK(hipEventCreate(&e0), "hipEventCreate");
    LBM_HIP_CHECK(hipEventCreate(&e1), "hipEventCreate");
    LBM_HIP_CHECK(hipEventCreate(&e2), "hipEventCreate");
    struct EvGuard {
        hipEvent_t* e;
        ~EvGuard() {
            for (int k = 0; k < 3; ++k) (void)hipEventDestroy(e[k]);
        }
    };
    hipEvent_t evs[3] = {e0, e1, e2};
    EvGuard guard{evs};

    // P_0 in both context lattices, then its wall slots into every other state:
    // the rest of them is written by the step that makes the state
    c->initialized = false;  // the lattices hold no resumable state from here on
    rc = launch_initialize<T, lbm::ST_NATIVE>(c);
    if (rc) return rc;
    rc = launch_walls<T, lbm::ST_NATIVE>(c, ckpt.data() + 1, ckpt.size() - 1, true);
    if (!rc) rc = launch_walls<T, lbm::ST_NATIVE>(c, tapes.data(), tapes.size(), true);
    if (rc) return rc;

    // forward with checkpoints
    LBM_HIP_CHECK(hipEventRecord(e0, c->stream), "hipEventRecord");
    void* fin = c->lat[1];
    for (int64_t m = 0; m < M; ++m) {
        const int64_t s0 = m * K;
        const int64_t len = std::min(K, T_steps - s0);
        void* const* const tape = tape_of(m);
        const void* src = ckpt[size_t(m)];
        for (int64_t j = 1; j <= len; ++j) {  // produce P_{s0 + j}
            void* dst;
            if (j == len)
                dst = m == M - 1 ? fin : ckpt[size_t(m + 1)];
            else
                dst = is_kept(m) ? tape[j - 1] : tape[(j - 1) % 2];
            rc = launch_compute<T, lbm::ST_NATIVE>(c, src, dst, 0, 0);
            if (rc) return rc;
            src = dst;
        }
    }
    LBM_HIP_CHECK(hipEventRecord(e1, c->stream), "hipEventRecord");

    lbm::AdjArgs<T> a{};
    a.grad_acc = grad_acc;
    a.partials = partials;
    a.n3 = c->n3;
    a.stride = c->stride;
    a.n = c->n;
    a.log2n = c->log2n;
    a.inv_tau = T(c->inv_tau);
    a.U = T(c->U);
    a.objective = cfg.objective;
    a.plane_z = cfg.plane_z;
    a.xcd_remap = c->cfg.xcd_remap >= 0 ? 1 : 0;
    {
        // number of FLUID/MOVING cells in the plane z = plane_z (all interior cells of that plane but the
        // boundary-layer ones); counted on the host
        int64_t np = 0;
        for (int32_t y = 0; y < c->n; ++y)
            for (int32_t x = 0; x < c->n; ++x)
                if (lbm::is_store_macro(lbm::cell_type(x, y, cfg.plane_z, c->n))) ++np;
        a.plane_scale = np > 0 ? 1.0 / double(np) : 0.0;
    }
    auto adj_step = [&](const void* P, const void* Lnext, void* Lprev, int seed, int first) -> int {
        a.P = static_cast<const T*>(P);
        a.Lnext = static_cast<const T*>(Lnext);
        a.Lprev = static_cast<T*>(Lprev);
        a.seed = seed;
        a.first = first;
        if (vec && V == 2) {
            if constexpr (sizeof(T) == 4)
                hipLaunchKernelGGL((lbm::lbm_adjoint_vec<T, 2>), dim3(unsigned(nblocks)), dim3(block), 0, c->stream,
                                   a);
        } else if (vec)
            hipLaunchKernelGGL((lbm::lbm_adjoint_vec<T, 1>), dim3(unsigned(nblocks)), dim3(block), 0, c->stream, a);
        else
            hipLaunchKernelGGL((lbm::lbm_adjoint_step<T>), dim3(unsigned(nblocks)), dim3(block), 0, c->stream, a);
        LBM_HIP_CHECK(hipGetLastError(), "adjoint step launch");
        return LBM_OK;
    };

    // seed: lambda_T from the objective evaluated on P_T
    int cur = 0;
    rc = adj_step(fin, nullptr, lam[cur], 1, T_steps == 0 ? 1 : 0);
    if (rc) return rc;
    // reverse sweep
    for (int64_t m = M - 1; m >= 0; --m) {
        const int64_t s0 = m * K;
        const int64_t len = std::min(K, T_steps - s0);
        void* const* const tape = tape_of(m);
        if (!is_kept(m)) {  // recompute P_{s0+1} .. P_{s0+len-1}
            const void* src = ckpt[size_t(m)];
            for (int64_t j = 1; j < len; ++j) {
                rc = launch_compute<T, lbm::ST_NATIVE>(c, src, tape[j - 1], 0, 0);
                if (rc) return rc;
                src = tape[j - 1];
            }
        }
        for (int64_t j = len - 1; j >= 0; --j) {  // step k = s0 + j reads P_k
            const void* Pk = (j == 0) ? ckpt[size_t(m)] : tape[j - 1];
            rc = adj_step(Pk, lam[cur], lam[1 - cur], 0, (s0 + j == 0) ? 1 : 0);
            if (rc) return rc;
            cur = 1 - cur;
            if (staged && grad_acc && (s0 + j) % lbm::ADJ_FLUSH == 0) {
                const int64_t n = 3 * c->n3;
                hipLaunchKernelGGL(lbm::lbm_adjoint_flush, dim3(unsigned((n + 255) / 256)), dim3(256), 0, c->stream,
                                   reinterpret_cast<float*>(grad_acc), grad_g, n);
                LBM_HIP_CHECK(hipGetLastError(), "adjoint flush launch");
            }
        }
    }
    hipLaunchKernelGGL(lbm::lbm_adjoint_reduce, dim3(1), dim3(1024), 0, c->stream, partials, nblocks, acc);
    LBM_HIP_CHECK(hipGetLastError(), "adjoint reduce launch");
    LBM_HIP_CHECK(hipEventRecord(e2, c->stream), "hipEventRecord");

    double h[3];
    rc = copy_to_host(c, h, acc, sizeof h);
    if (!rc && grad_g_host) rc = copy_to_host(c, grad_g_host, grad_g, size_t(3 * c->n3) * sizeof(double));
    if (rc) return rc;
    float fms = 0.f, ams = 0.f;
    LBM_HIP_CHECK(hipEventElapsedTime(&fms, e0, e1), "hipEventElapsedTime");
    LBM_HIP_CHECK(hipEventElapsedTime(&ams, e1, e2), "hipEventElapsedTime");
    const double om = c->inv_tau;
    res->objective = h[2];
    res->d_velocity = h[0];
    res->d_viscosity = h[1] * (-3.0 * om * om);  // omega = 1 / (3 nu + 1/2)
    res->forward_ms = double(fms);
    res->adjoint_ms = double(ams);
    res->device_bytes = device_bytes;
    res->checkpoints = M;
    res->segment = K;
    return LBM_OK;
}

}  // namespace

extern "C" {

int lbm_set_force(lbm_ctx* c, const void* force) {
    if (!c) return fail(LBM_ERR_INVALID, "null context");
    int rc = set_device(c);
    if (rc) return rc;
    LBM_HIP_CHECK(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    if (!force) {
        g_pool.give(c->cfg.device, c->force, size_t(3 * c->n3) * c->tsize);
        c->force = nullptr;
        return LBM_OK;
    }
    const size_t bytes = size_t(3 * c->n3) * c->tsize;
    if (!c->force) {
        rc = pool_alloc(c, &c->force, bytes, "body force");
        if (rc) return rc;
    }
    LBM_HIP_CHECK(hipMemcpyAsync(c->force, force, bytes, hipMemcpyHostToDevice, c->stream), "hipMemcpyAsync H2D");
    LBM_HIP_CHECK(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    return LBM_OK;
}

int lbm_adjoint(lbm_ctx* c, const lbm_adjoint_config* cfg, lbm_adjoint_result* res, double* grad_force) {
    if (!cfg || !res) return fail(LBM_ERR_INVALID, "null argument");
    // the layout check comes first: it needs no device
    if (cfg->struct_size != sizeof(lbm_adjoint_config))
        return fail(LBM_ERR_INVALID, "lbm_adjoint_config.struct_size is " + std::to_string(cfg->struct_size) +
                                         ", this library's lbm_adjoint_config has " +
                                         std::to_string(sizeof(lbm_adjoint_config)) +
                                         " bytes (set it to sizeof(lbm_adjoint_config), e.g. with "
                                         "LBM_ADJOINT_CONFIG_INIT)");
    if (!c) return fail(LBM_ERR_INVALID, "null context");
    int rc = set_device(c);
    if (rc) return rc;
    if (c->cfg.storage != LBM_STORE_NATIVE) return fail(LBM_ERR_INVALID, "the adjoint needs native storage");
    if (cfg->steps < 1) return fail(LBM_ERR_INVALID, "adjoint needs steps >= 1");
    if (cfg->objective != LBM_OBJECTIVE_KINETIC_ENERGY && cfg->objective != LBM_OBJECTIVE_MEAN_UX_PLANE)
        return fail(LBM_ERR_INVALID, "unknown objective");
    if (cfg->objective == LBM_OBJECTIVE_MEAN_UX_PLANE && (cfg->plane_z < 1 || cfg->plane_z > c->n - 2))
        return fail(LBM_ERR_INVALID, "plane_z must be an interior plane");
    if (c->n < 4) return fail(LBM_ERR_INVALID, "the adjoint needs dim >= 4");
    std::memset(res, 0, sizeof *res);
    if (c->cfg.precision == LBM_F64) return run_adjoint<double>(c, *cfg, res, grad_force);
    return run_adjoint<float>(c, *cfg, res, grad_force);
}

}  // extern "C"
