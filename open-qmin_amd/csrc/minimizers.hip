// Adam, Nesterov accelerated gradient and online L-BFGS on the device.
//
// An Adam or Nesterov iteration is one lattice pass (the fused and boundary
// passes in mode kAdamStep / kNesterovStep, step_kernels.hip): each site's
// force, then the minimizer's update of that site, written to the other state
// set.  An L-BFGS iteration is the shared force pass (force mode) and two
// streaming kernels over the 5 n components of Q, F and the minimizer's own
// vectors (same plane layout as Q).  Every pass reduces the dot products it
// needs into per-work-group partials; a one-work-group kernel sums them in a
// fixed order and finishes the minimizer's scalar logic in device memory (step
// coefficients, forceMax, the stopping test).  (A separate kernel, not a
// last-work-group pattern: the device-wide fences that pattern needs write back
// each XCD's L2, which the streaming kernel has just filled.)  A batch of
// iterations is therefore queued without host round trips, every kernel after
// the stopping test is a no-op, and the host reads the control block once per
// batch.
//
// Arithmetic follows the reference CPU steps: energyMinimizerAdam.cpp:25-54,
// energyMinimizerNesterovAG.cpp:70-92 and energyMinimizerLoLBFGS.cpp:104-193.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "qmin_internal.h"

namespace qmin {
namespace {

constexpr int kVecThreads = 256;

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Iteration bookkeeping shared by the three minimizers (thread 0 of the last
// work-group): count, forceMax, trace, and the loop test of minimize().
__device__ void finish_iteration(Ctrl* ctrl, double forceMax, double fc, double* trace) {
    const int it = ctrl->iterations + 1;
    ctrl->iterations = it;
    ctrl->forceMax = forceMax;
    if (trace && ctrl->traceLen < ctrl->traceCap) {
        trace[ctrl->traceLen] = forceMax;
        ctrl->traceLen += 1;
    }
    if (isnan(forceMax)) ctrl->nanFlag = 1;
    ctrl->done = !(it < ctrl->maxIter && forceMax > fc);
}

struct Common {
    Ctrl* ctrl;
    double* partials;
    double* trace;      // [traceCap] forceMax per iteration
    double fc, ndof;
    long long len;      // 5 n
};

// ---------------------------------------------------------------- online L-BFGS
// The direction of an iteration is a combination of the forces and the history,
// p = F + sum_t cy_t y_t + sum_t cs_t s_t.  The two-loop recursion
// (energyMinimizerLoLBFGS.cpp:117-163) that fixes the coefficients needs only
// scalar products: s_t.y_u and y_t.y_u, kept between iterations with the new
// pair's rows replaced, and s_t.F and y_t.F.  So one pass over the history takes
// the products, one work-group runs the recursion on them, and one pass forms
// the direction and takes the step: at m = 8, 39 vectors read or written per
// iteration instead of the 72 of one streaming pass per two-loop stage, and 3
// launches beside the force's instead of 34.  At 100 x 96 x 104 in FP64, m = 8:
// 0.38 ms per iteration against 0.66 (passes 144 and 148 us, 5.3 and 5.7 TB/s;
// recursion 13 us).
//
// Device scalars: SY[u m + t] = s_t.y_u, YY[u m + t] = y_t.y_u, the
// coefficients of the next step, and the recursion's work space (the products,
// sp, yp, alpha, F.F).
struct LbLayout {
    int m;
    __host__ __device__ int SY(int u, int t) const { return u * m + t; }
    __host__ __device__ int YY(int u, int t) const { return m * m + u * m + t; }
    __host__ __device__ int CY(int t) const { return 2 * m * m + t; }
    __host__ __device__ int CS(int t) const { return 2 * m * m + m + t; }
    __host__ __device__ int work() const { return 2 * m * m + 2 * m; }
    __host__ __device__ int workSize() const { return 8 * m + 1; }
    __host__ __device__ int size() const { return work() + workSize(); }
};

constexpr int kLbBlock = 8;                       // slots whose products one launch takes
constexpr int kLbDots = 5 * kLbBlock + 1;         // products per launch
constexpr int kLbBlocks = 512;                    // work-groups of the passes over the history at most

template <typename R>
struct LbArgs {
    R* hist;            // s_0 .. s_{m-1}, y_0 .. y_{m-1}, stride components apart
    long long stride;
    const R* f;
    const R* p;         // the forces the products were taken of: f, but for the first step of a later call
    R* q;
    double eta;
    int m, c, t0;       // memory, the slot being replaced, first slot of this launch's products
    double* scal;
    Common c0;
};

// y_c = y_c - F (the move stored the old forces there, :178-188), then the
// products of the new pair and of F with the slots t0 .. t0 + 7, and F.F.
// Bound by HBM: 2 m + 3 vectors.
template <typename R>
__global__ void __launch_bounds__(kVecThreads) lb_dots_kernel(LbArgs<R> A) {
    if (A.c0.ctrl->done) return;
    double acc[kLbDots];
#pragma unroll
    for (int k = 0; k < kLbDots; ++k) acc[k] = 0;
    const R* s0 = A.hist;
    const R* y0 = A.hist + A.m * A.stride;
    R* yc = A.hist + (A.m + A.c) * A.stride;
    const R* sc = A.hist + A.c * A.stride;
    const int count = min(kLbBlock, A.m - A.t0);
    auto site = [&](long long i, auto width) {
        constexpr int W = decltype(width)::value;
        using V = R __attribute__((ext_vector_type(W)));
        auto at = [&](const R* p) { return *reinterpret_cast<const V*>(p + i); };
        const V f = at(A.f), so = at(sc);
        V yn = at(yc);
        if (A.t0 == 0) {
            yn = yn - f;
            *reinterpret_cast<V*>(yc + i) = yn;
        }
        V sv[kLbBlock], yv[kLbBlock];
#pragma unroll
        for (int k = 0; k < kLbBlock; ++k)
            if (k < count) {
                sv[k] = at(s0 + (A.t0 + k) * A.stride);
                yv[k] = A.t0 + k == A.c ? yn : at(y0 + (A.t0 + k) * A.stride);
            }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const double fd = double(f[w]), yd = double(yn[w]), sd = double(so[w]);
            acc[kLbDots - 1] += fd * fd;
#pragma unroll
            for (int k = 0; k < kLbBlock; ++k)
                if (k < count) {
                    const double a = double(sv[k][w]), b = double(yv[k][w]);
                    acc[5 * k + 0] += a * fd;
                    acc[5 * k + 1] += b * fd;
                    acc[5 * k + 2] += a * yd;
                    acc[5 * k + 3] += b * yd;
                    acc[5 * k + 4] += sd * b;
                }
        }
    };
    const long long pairs = A.c0.len / 2, step = (long long)gridDim.x * kVecThreads;
    for (long long j = (long long)blockIdx.x * kVecThreads + threadIdx.x; j < pairs; j += step)
        site(2 * j, std::integral_constant<int, 2>{});
    if ((A.c0.len & 1) && blockIdx.x == 0 && threadIdx.x == 0) site(A.c0.len - 1, std::integral_constant<int, 1>{});
    // work-group sums in a fixed order; partials[k][work-group]
    __shared__ double red[kVecThreads / 64][kLbDots];
#pragma unroll
    for (int k = 0; k < kLbDots; ++k) {
        const double v = wsum(acc[k]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = v;
    }
    __syncthreads();
    if (threadIdx.x < kLbDots) {
        double v = 0;
#pragma unroll
        for (int w = 0; w < kVecThreads / 64; ++w) v += red[w][threadIdx.x];
        A.c0.partials[((long long)(A.t0 / kLbBlock) * kLbDots + threadIdx.x) * kLbBlocks + blockIdx.x] = v;
    }
}

// Sums the products in a fixed order (a wave per product), replaces the new
// pair's rows of SY and YY, runs the two-loop recursion on the products (sp_t =
// s_t.p and yp_t = y_t.p as p grows), and ends the iteration.  Its length is
// that of the recursion's 2 m dependent steps: with LDS they read SY, YY and
// the work space from there (up to kLbLdsMemory slots), else from memory.
constexpr int kLbCoefThreads = 512;
constexpr int kLbLdsMemory = 32;
template <bool LDS>
__global__ void __launch_bounds__(kLbCoefThreads) lb_coef_kernel(Common c, double* scal, LbLayout lay, int slot,
                                                                int blocks) {
    __shared__ double lds[LDS ? 2 * kLbLdsMemory * kLbLdsMemory + 8 * kLbLdsMemory + 1 : 1];
    Ctrl* ctrl = c.ctrl;
    if (ctrl->done) return;
    const int m = lay.m, tid = threadIdx.x, mm = m * m;
    double* SY = LDS ? lds : scal;
    double* YY = SY + mm;
    double* dots = LDS ? lds + 2 * mm : scal + lay.work();
    double* sp = dots + 5 * m;
    double* yp = sp + m;
    double* alpha = yp + m;
    double* ff = alpha + m;
    if constexpr (LDS)
        for (int k = tid; k < 2 * mm; k += kLbCoefThreads) lds[k] = scal[k];
    for (int k = tid >> 6; k <= 5 * m; k += kLbCoefThreads / 64) {
        const int block = k == 5 * m ? 0 : k / (5 * kLbBlock), row = k == 5 * m ? kLbDots - 1 : k % (5 * kLbBlock);
        const double* part = c.partials + ((long long)block * kLbDots + row) * kLbBlocks;
        double v = 0;
#pragma unroll 8
        for (int j = tid & 63; j < blocks; j += 64) v += part[j];
        v = wsum(v);
        if ((tid & 63) == 0) *(k == 5 * m ? ff : dots + k) = v;
    }
    __syncthreads();
    for (int t = tid; t < m; t += kLbCoefThreads) {
        sp[t] = dots[5 * t + 0];
        yp[t] = dots[5 * t + 1];
        const double sy = dots[5 * t + 2], yy = dots[5 * t + 3], ys = dots[5 * t + 4];
        SY[slot * m + t] = sy;
        YY[slot * m + t] = yy;
        YY[t * m + slot] = yy;
        SY[t * m + slot] = ys;
        if constexpr (LDS) {
            scal[lay.SY(slot, t)] = sy;
            scal[lay.YY(slot, t)] = yy;
            scal[lay.YY(t, slot)] = yy;
            scal[lay.SY(t, slot)] = ys;
        }
    }
    __syncthreads();
    // newest slot first (:117-131); a pair with s.y = 0 is skipped
    for (int i = 0; i < m; ++i) {
        const int t = (slot - i + m) % m;
        const double sy = SY[t * m + t];
        const double a = sy != 0 ? sp[t] / sy : 0.0;
        __syncthreads();
        for (int u = tid; u < m; u += kLbCoefThreads) {
            sp[u] -= a * SY[t * m + u];
            yp[u] -= a * YY[t * m + u];
        }
        if (tid == 0) alpha[i] = a;
        __syncthreads();
    }
    // step 3 (:133-142): p += (s.y / y.y) y of the newest slot
    const double yy = YY[slot * m + slot];
    const double k3 = yy != 0 ? SY[slot * m + slot] / yy : 0.0;
    for (int u = tid; u < m; u += kLbCoefThreads) yp[u] += k3 * YY[slot * m + u];
    __syncthreads();
    // oldest first (:145-163)
    for (int i = m - 1; i >= 0; --i) {
        const int t = (slot - i + m) % m;
        const double sy = SY[t * m + t];
        const double d = sy != 0 ? alpha[i] - yp[t] / sy : 0.0;
        __syncthreads();
        for (int u = tid; u < m; u += kLbCoefThreads) yp[u] += d * SY[u * m + t];
        if (tid == 0) {
            scal[lay.CS(t)] = d;
            scal[lay.CY(t)] = (i == 0 ? k3 : 0.0) - alpha[i];
        }
        __syncthreads();
    }
    if (tid == 0) finish_iteration(ctrl, sqrt(*ff) / c.ndof, c.fc, c.trace);
}

// p = F + sum_t cy_t y_t + sum_t cs_t s_t in FP64; then s_c = eta p, y_c = F (the old forces), Q += s_c (:158-176).  Runs from the end of
// the vectors to their start: the last of what the products' pass read is still
// in the memory-side cache.  Bound by HBM: 2 m + 5 vectors.
template <typename R>
__global__ void __launch_bounds__(kVecThreads) lb_move_kernel(LbArgs<R> A) {
    if (A.c0.ctrl->done) return;
    const LbLayout lay{A.m};
    auto site = [&](long long i, auto width) {
        constexpr int W = decltype(width)::value;
        using V = R __attribute__((ext_vector_type(W)));
        auto at = [&](const R* p) { return *reinterpret_cast<const V*>(p + i); };
        const V f = at(A.f), pv = at(A.p), q = at(A.q);
        double p[W];
#pragma unroll
        for (int w = 0; w < W; ++w) p[w] = double(pv[w]);
        for (int t0 = 0; t0 < A.m; t0 += kLbBlock) {
            V sv[kLbBlock], yv[kLbBlock];
#pragma unroll
            for (int k = 0; k < kLbBlock; ++k)
                if (t0 + k < A.m) {
                    sv[k] = at(A.hist + (t0 + k) * A.stride);
                    yv[k] = at(A.hist + (A.m + t0 + k) * A.stride);
                }
#pragma unroll
            for (int k = 0; k < kLbBlock; ++k)
                if (t0 + k < A.m) {
                    const double cy = A.scal[lay.CY(t0 + k)], cs = A.scal[lay.CS(t0 + k)];
#pragma unroll
                    for (int w = 0; w < W; ++w) p[w] += cy * double(yv[k][w]) + cs * double(sv[k][w]);
                }
        }
        V s;
#pragma unroll
        for (int w = 0; w < W; ++w) s[w] = R(A.eta * p[w]);
        *reinterpret_cast<V*>(A.hist + A.c * A.stride + i) = s;
        *reinterpret_cast<V*>(A.hist + (A.m + A.c) * A.stride + i) = f;
        *reinterpret_cast<V*>(A.q + i) = q + s;
    };
    const long long pairs = A.c0.len / 2, step = (long long)gridDim.x * kVecThreads;
    if ((A.c0.len & 1) && blockIdx.x == 0 && threadIdx.x == 0) site(A.c0.len - 1, std::integral_constant<int, 1>{});
    for (long long j = pairs - 1 - ((long long)blockIdx.x * kVecThreads + threadIdx.x); j >= 0; j -= step)
        site(2 * j, std::integral_constant<int, 2>{});
}

// ---------------------------------------------------------------- finalize
enum FinOp { kFinAdam, kFinNesterov };

struct FinArgs {
    int op;
    int blocks;       // partial-sum slots of the lattice passes to sum (3 doubles each, the first |F|^2)
    double b1, b2;    // Adam
    int scheduled;    // Nesterov
    double* scal;
    Common c;
};

// One work-group: fixed-order sum of the lattice passes' partials of |F|^2, then
// the minimizer's scalar step in thread 0 and the flip to the state set that
// the passes wrote.
__global__ void __launch_bounds__(kVecThreads) vec_finalize_kernel(FinArgs A) {
    __shared__ double red[kVecThreads / 64];
    Ctrl* ctrl = A.c.ctrl;
    if (ctrl->done) return;
    double tot = 0;
    for (int j = threadIdx.x; j < A.blocks; j += kVecThreads) tot += A.c.partials[3LL * j];
    tot = wsum(tot);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = tot;
    __syncthreads();
    if (threadIdx.x != 0) return;
    tot = 0;
#pragma unroll
    for (int w = 0; w < kVecThreads / 64; ++w) tot += red[w];
    double* scal = A.scal;
    if (A.op == kFinAdam) {
        // beta^t advances once per executed step (energyMinimizerAdam.cpp:52-53)
        scal[0] = scal[0] * A.b1;
        scal[1] = scal[1] * A.b2;
    } else {
        // the same lambda and momentum the step kernel computed from scal[0]
        const double oldLambda = scal[0];
        const double lambda = 0.5 * (1.0 + sqrt(1.0 + 4.0 * oldLambda * oldLambda));
        const double gamma = (1 - oldLambda) / lambda;
        if (A.scheduled) scal[1] = 1. + gamma;
        scal[0] = lambda;
    }
    finish_iteration(ctrl, sqrt(tot) / A.c.ndof, A.c.fc, A.c.trace);
    ctrl->cur ^= 1;
}

}  // namespace
}  // namespace qmin

using namespace qmin;

// ------------------------------------------------------------------ host side

// Device state common to the three minimizers: vectors of 5 n reals bound to
// one lattice, scalars, partial sums and the forceMax trace.
struct VecMinimizer {
    uint64_t bound = 0;   // serial of the lattice the vectors belong to (0: none)
    long long boundN = 0;
    int boundPrecision = -1;
    std::vector<void*> vecs;     // in one allocation, stride reals apart
    long long stride = 0;
    double* dScal = nullptr;
    int scalCount = 0;
    double* dPartials = nullptr;
    double* dTrace = nullptr;
    int dTraceCap = 0;
    int traceCap = 0;
    std::vector<double> trace;
    int iterations = 0, maxIter = 1000;
    double forceMax = 100.0, fc = 1e-12;
    int converged = 0, nan = 0;

    ~VecMinimizer() {
        release();
        if (dTrace) (void)hipFree(dTrace);
    }
    // drops the device history (the trace buffer stays)
    void release() {
        if (!vecs.empty()) (void)hipFree(vecs[0]);
        vecs.clear();
        if (dScal) (void)hipFree(dScal);
        if (dPartials) (void)hipFree(dPartials);
        dScal = nullptr;
        dPartials = nullptr;
        bound = 0;
        boundN = 0;
        boundPrecision = -1;
    }
    bool needs_bind(const qm_lattice* L) const {
        return bound != L->serial || boundN != L->n || boundPrecision != L->precision;
    }
    // (re)allocates nv zeroed vectors, nscal zeroed scalars and nparts partial
    // sums of its own for lattice L
    int bind(qm_lattice* L, int nv, int nscal, size_t nparts = 0) {
        release();
        const size_t align = 256 / L->realSize;   // each vector on a 256-byte boundary
        stride = (long long)((5 * (size_t)L->n + align - 1) / align * align);
        const size_t bytes = (size_t)stride * L->realSize;
        char* base = nullptr;
        if (hipMalloc(&base, nv * bytes) != hipSuccess)
            return fail(QM_ENOMEM, "minimizer vectors: out of device memory");
        for (int k = 0; k < nv; ++k) vecs.push_back(base + k * bytes);
        HIP_TRY(hipMemsetAsync(base, 0, nv * bytes, L->stream));
        HIP_TRY(hipMalloc(&dScal, std::max(nscal, 1) * sizeof(double)));
        HIP_TRY(hipMemsetAsync(dScal, 0, std::max(nscal, 1) * sizeof(double), L->stream));
        scalCount = nscal;
        if (nparts) HIP_TRY(hipMalloc(&dPartials, nparts * sizeof(double)));
        bound = L->serial;
        boundN = L->n;
        boundPrecision = L->precision;
        return QM_OK;
    }
    int ensure_trace() {
        if (traceCap > dTraceCap) {
            if (dTrace) HIP_TRY(hipFree(dTrace));
            HIP_TRY(hipMalloc(&dTrace, (size_t)traceCap * sizeof(double)));
            dTraceCap = traceCap;
        }
        return QM_OK;
    }
    Common common(const qm_lattice* L) const {
        Common c{};
        c.ctrl = L->dCtrl;
        c.partials = dPartials;
        c.trace = traceCap > 0 ? dTrace : nullptr;
        c.fc = fc;
        c.ndof = (double)L->n;
        c.len = 5 * L->n;
        return c;
    }
    int set_scalars(const qm_lattice* L, const double* v, int count, int offset = 0) {
        HIP_TRY(hipMemcpyAsync(dScal + offset, v, count * sizeof(double), hipMemcpyHostToDevice, L->stream));
        return QM_OK;
    }
    // the finalize kernel for a lattice pass of `blocks` partial-sum slots
    int finalize(const qm_lattice* L, FinArgs a, long long blocks) const {
        a.blocks = (int)blocks;
        a.scal = dScal;
        a.c = common(L);
        a.c.partials = L->dPartials;
        vec_finalize_kernel<<<1, kVecThreads, 0, L->stream>>>(a);
        HIP_TRY(hipGetLastError());
        return QM_OK;
    }
    int get_scalars(const qm_lattice* L, double* v, int count, int offset = 0) {
        HIP_TRY(hipMemcpyAsync(v, dScal + offset, count * sizeof(double), hipMemcpyDeviceToHost, L->stream));
        HIP_TRY(hipStreamSynchronize(L->stream));
        return QM_OK;
    }
};

// Starts a minimize call: FIRE's pending velocity is made concrete (it is kept
// in the same state set), the control block is set for this minimizer.
static int begin_run(VecMinimizer& s, qm_lattice* L, const qm_ldg* f, bool done) {
    if (int rc = prepare(L, f)) return rc;
    if (int rc = materialize(L)) return rc;
    if (int rc = s.ensure_trace()) return rc;
    if (int rc = sync_ctrl_to_host(L)) return rc;
    Ctrl& c = L->hCtrl;
    c.done = done ? 1 : 0;
    c.iterations = s.iterations;
    c.maxIter = s.maxIter;
    c.nanFlag = 0;
    c.traceLen = 0;
    c.traceCap = s.traceCap;
    c.forceMax = s.forceMax;
    return push_ctrl(L);
}

// Queues batches of iterations until the control block reports done.
template <typename Enqueue>
static int drive(VecMinimizer& s, qm_lattice* L, Enqueue&& enqueue) {
    const int batch = L->n >= (1 << 22) ? 16 : 64;
    int queued = 0;
    while (!L->hCtrl.done) {
        int todo = std::min(batch, s.maxIter - (s.iterations + queued));
        if (todo <= 0) todo = 1;
        for (int k = 0; k < todo; ++k) {
            if (int rc = enqueue(s.iterations + queued)) return rc;
            ++queued;
        }
        if (int rc = sync_ctrl_to_host(L)) return rc;
        // iterations the device actually ran: the rest were skipped
        queued = L->hCtrl.iterations - s.iterations;
    }
    const Ctrl& h = L->hCtrl;
    s.iterations = h.iterations;
    s.forceMax = h.forceMax;
    s.nan = h.nanFlag;
    s.converged = !h.nanFlag && h.forceMax <= s.fc;
    if (s.traceCap > 0 && h.traceLen > 0) {
        const size_t old = s.trace.size();
        s.trace.resize(old + (size_t)h.traceLen);
        HIP_TRY(copy_on(L, s.trace.data() + old, s.dTrace, (size_t)h.traceLen * sizeof(double),
                          hipMemcpyDeviceToHost));
    }
    if (h.nanFlag) return fail(QM_ENAN, "minimizer produced a NaN force norm");
    return QM_OK;
}

// Drives Adam or Nesterov.  Nothing reads the forces of an iteration but the last,
// so only a pass that is known to be the last stores them (40 of the 201 B that
// an FP64 Nesterov pass would move per site); where the tolerance stopped the run
// before its limit, they are computed again from the Q they belong to.  A run of
// a few iterations stores them always, and one with a tolerance in its first two,
// after which the passes have saved what that computation takes: Nesterov, L1..L3,
// 150^3 in FP64, stopped after one iteration 817 us, with the computation 852.  Without
// stores Nesterov, L1..L3, 192 x 150 x 130 in FP64 takes 158 us per iteration,
// with them 190.
constexpr int kFewIterations = 4, kFirstIterations = 2;
template <typename Enqueue>
static int drive_steps(VecMinimizer& s, qm_lattice* L, const qm_ldg* f, Enqueue&& enqueue) {
    const int begin = s.iterations;
    const int first = s.maxIter - begin <= kFewIterations ? kFewIterations : s.fc > 0 ? kFirstIterations : 0;
    const int rc =
        drive(s, L, [&](int iteration) { return enqueue(iteration - begin < first || iteration + 1 >= s.maxIter); });
    if (s.iterations - begin > first && s.iterations < s.maxIter)
        if (int rc2 = last_step_force(L, f)) return rc ? rc : rc2;
    return rc;
}

template <typename R>
static R* rp(void* p) {
    return static_cast<R*>(p);
}

// ------------------------------------------------------------------ Adam
struct qm_adam : VecMinimizer {
    // setAdamParameters defaults (energyMinimizerAdam.h:16-25)
    double b1 = 0.9, b2 = 0.99, eps = 1e-8, dt = 1e-4;
    double b1t = 0.9, b2t = 0.99;
};

static int adam_enqueue(qm_adam* m, qm_lattice* L, const qm_ldg* f, bool storeF) {
    StepArgs st{};
    st.m = m->vecs[0];
    st.v = m->vecs[1];
    st.scal = m->dScal;
    st.b1 = m->b1;
    st.b2 = m->b2;
    st.eps = m->eps;
    st.dt = m->dt;
    long long slots = 0;
    if (int rc = step_pass(L, f, kAdamStep, st, storeF, &slots)) return rc;
    FinArgs fa{};
    fa.op = kFinAdam;
    fa.b1 = m->b1;
    fa.b2 = m->b2;
    return m->finalize(L, fa, slots);
}

extern "C" {

int qm_adam_create(qm_adam** out) {
    if (!out) return fail(QM_EINVAL, "null output handle");
    *out = new qm_adam;
    (*out)->forceMax = 110.0;
    return QM_OK;
}

int qm_adam_destroy(qm_adam* m) {
    delete m;
    return QM_OK;
}

int qm_adam_set_parameters(qm_adam* m, double beta1, double beta2, double eps, double dt, double forceCutoff) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->b1 = beta1;
    m->b1t = beta1;
    m->b2 = beta2;
    m->b2t = beta2;
    m->eps = eps;
    m->dt = dt;
    m->fc = forceCutoff;
    return QM_OK;
}

int qm_adam_set_max_iterations(qm_adam* m, int maxIterations) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->maxIter = maxIterations;
    return QM_OK;
}

int qm_adam_minimize(qm_adam* m, qm_ldg* f, qm_lattice* L) {
    if (!m || !f || !L) return fail(QM_EINVAL, "null handle");
    if (m->needs_bind(L)) {
        // initializeFromModel (energyMinimizerAdam.cpp:9-23): zero moments, iteration 0
        if (int rc = m->bind(L, 2, 2)) return rc;
        m->iterations = 0;
        m->b1t = m->b1;
        m->b2t = m->b2;
    }
    m->forceMax = 110.0;
    if (int rc = begin_run(*m, L, f, m->iterations >= m->maxIter)) return rc;
    // the iterations alternate the state sets and leave U alone
    if (int rc = share_velocity(L)) return rc;
    const double sc[2] = {m->b1t, m->b2t};
    if (int rc = m->set_scalars(L, sc, 2)) return rc;
    int rc = drive_steps(*m, L, f, [&](bool storeF) { return adam_enqueue(m, L, f, storeF); });
    double back[2];
    if (int r2 = m->get_scalars(L, back, 2)) return r2;
    m->b1t = back[0];
    m->b2t = back[1];
    return rc;
}

int qm_adam_get_state(const qm_adam* m, int* iterations, double* forceMax) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    if (iterations) *iterations = m->iterations;
    if (forceMax) *forceMax = m->forceMax;
    return QM_OK;
}

}  // extern "C"

// ------------------------------------------------------------------ Nesterov
struct qm_nesterov : VecMinimizer {
    // setNesterovAGParameters defaults (energyMinimizerNesterovAG.h:22-27)
    double dt = 1e-4, mu = 0.01;
    double mu0 = 0.01;   // mu as set: the scheduled momentum restarts from it
    double lambda = 1.0;
    int scheduled = 0;
};

static int nesterov_enqueue(qm_nesterov* m, qm_lattice* L, const qm_ldg* f, bool storeF) {
    StepArgs st{};
    st.m = m->vecs[0];
    st.scal = m->dScal;
    st.dt = m->dt;
    st.scheduled = m->scheduled;
    long long slots = 0;
    if (int rc = step_pass(L, f, kNesterovStep, st, storeF, &slots)) return rc;
    FinArgs fa{};
    fa.op = kFinNesterov;
    fa.scheduled = m->scheduled;
    return m->finalize(L, fa, slots);
}

extern "C" {

int qm_nesterov_create(qm_nesterov** out) {
    if (!out) return fail(QM_EINVAL, "null output handle");
    *out = new qm_nesterov;
    return QM_OK;
}

int qm_nesterov_destroy(qm_nesterov* m) {
    delete m;
    return QM_OK;
}

int qm_nesterov_set_parameters(qm_nesterov* m, double dt, double mu, double forceCutoff, int scheduledMomentum) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->dt = dt;
    m->mu = mu;
    m->mu0 = mu;
    m->fc = forceCutoff;
    m->scheduled = scheduledMomentum != 0;
    return QM_OK;
}

int qm_nesterov_set_max_iterations(qm_nesterov* m, int maxIterations) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->maxIter = maxIterations;
    return QM_OK;
}

int qm_nesterov_minimize(qm_nesterov* m, qm_ldg* f, qm_lattice* L) {
    if (!m || !f || !L) return fail(QM_EINVAL, "null handle");
    m->forceMax = 110.0;
    // a new lattice (or precision) starts a new run: iteration 0, momentum as set
    const bool rebind = m->needs_bind(L);
    if (rebind) {
        if (int rc = m->bind(L, 1, 2)) return rc;
        m->iterations = 0;
        m->lambda = 1.0;
        m->mu = m->mu0;
    }
    if (int rc = begin_run(*m, L, f, m->iterations >= m->maxIter)) return rc;
    // the iterations alternate the state sets and leave U alone
    if (int rc = share_velocity(L)) return rc;
    if (rebind) {
        // initializeFromModel (energyMinimizerNesterovAG.cpp:31-37): the
        // alternate sequence starts as a copy of the positions
        HIP_TRY(hipMemcpyAsync(m->vecs[0], L->dSet[L->hCtrl.cur], 5 * (size_t)L->n * L->realSize,
                               hipMemcpyDeviceToDevice, L->stream));
    }
    const double sc[2] = {m->lambda, m->mu};
    if (int rc = m->set_scalars(L, sc, 2)) return rc;
    int rc = drive_steps(*m, L, f, [&](bool storeF) { return nesterov_enqueue(m, L, f, storeF); });
    double back[2];
    if (int r2 = m->get_scalars(L, back, 2)) return r2;
    m->lambda = back[0];
    m->mu = back[1];
    return rc;
}

int qm_nesterov_get_state(const qm_nesterov* m, int* iterations, double* forceMax) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    if (iterations) *iterations = m->iterations;
    if (forceMax) *forceMax = m->forceMax;
    return QM_OK;
}

}  // extern "C"

// ------------------------------------------------------------------ online L-BFGS
struct qm_lolbfgs : VecMinimizer {
    // setLoLBFGSParameters defaults (energyMinimizerLoLBFGS.h:29-45); the memory
    // only grows, starting from the constructor's 5
    int m = 5;
    double dt = 1e-4, c = 1.0, tau = 10.0;
    int scheduled = 0;
    int cur = 0;   // currentIterationInMLoop
    bool fresh = true;   // p must be (re)started from the forces: new or re-initialised history
    // vecs: [0 .. m-1] s, [m .. 2m-1] y, [2m] the direction a call ended with: p = F,
    // of which the coefficients kept for the next call are
};

template <typename R>
static int lb_enqueue(qm_lolbfgs* M, qm_lattice* L, const qm_ldg* f, int iteration, bool first) {
    const int m = M->m, c = M->cur;
    const StateSet<R> st = state_set<R>(L, L->hCtrl.cur);
    LbArgs<R> a{};
    a.hist = rp<R>(M->vecs[0]);
    a.stride = M->stride;
    a.f = st.f;
    a.p = first ? rp<R>(M->vecs[2 * m]) : st.f;
    a.q = st.q;
    a.m = m;
    a.c = c;
    a.scal = M->dScal;
    a.c0 = M->common(L);
    if (M->fresh) {
        // step 1 (energyMinimizerLoLBFGS.cpp:107-114): p = F(Q); the history is
        // empty and its coefficients are zero.  A history re-initialised after
        // iterations also starts here.
        M->fresh = false;
        if (int rc = force_pass(L, f, true)) return rc;
        a.p = st.f;
    }
    const long long pairs = (a.c0.len + 1) / 2;
    const int blocks = (int)std::min<long long>((pairs + kVecThreads - 1) / kVecThreads, kLbBlocks);
    // update step: eta as minimize() sets it (energyMinimizerLoLBFGS.cpp:203-209)
    a.eta = M->scheduled ? M->tau / (M->tau + iteration) * M->dt : M->dt;
    lb_move_kernel<R><<<blocks, kVecThreads, 0, L->stream>>>(a);
    HIP_TRY(hipGetLastError());
    if (int rc = force_pass(L, f, true)) return rc;
    for (a.t0 = 0; a.t0 < m; a.t0 += kLbBlock) {
        lb_dots_kernel<R><<<blocks, kVecThreads, 0, L->stream>>>(a);
        HIP_TRY(hipGetLastError());
    }
    if (m <= kLbLdsMemory)
        lb_coef_kernel<true><<<1, kLbCoefThreads, 0, L->stream>>>(a.c0, M->dScal, LbLayout{m}, c, blocks);
    else
        lb_coef_kernel<false><<<1, kLbCoefThreads, 0, L->stream>>>(a.c0, M->dScal, LbLayout{m}, c, blocks);
    HIP_TRY(hipGetLastError());
    M->cur = (c + 1) % m;
    return QM_OK;
}

extern "C" {

int qm_lolbfgs_create(qm_lolbfgs** out) {
    if (!out) return fail(QM_EINVAL, "null output handle");
    *out = new qm_lolbfgs;
    return QM_OK;
}

int qm_lolbfgs_destroy(qm_lolbfgs* m) {
    delete m;
    return QM_OK;
}

int qm_lolbfgs_set_parameters(qm_lolbfgs* m, int memory, double dt, double c, double forceCutoff, double tau,
                              int scheduledMomentum) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->c = c;
    m->dt = dt;
    m->tau = tau;
    m->fc = forceCutoff;
    m->scheduled = scheduledMomentum != 0;
    if (memory > m->m) {
        // a larger memory re-initialises the history (energyMinimizerLoLBFGS.h:36-43)
        m->m = memory;
        m->release();
    }
    return QM_OK;
}

int qm_lolbfgs_set_max_iterations(qm_lolbfgs* m, int maxIterations) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    m->maxIter = maxIterations;
    return QM_OK;
}

int qm_lolbfgs_minimize(qm_lolbfgs* M, qm_ldg* f, qm_lattice* L) {
    if (!M || !f || !L) return fail(QM_EINVAL, "null handle");
    if (M->needs_bind(L)) {
        // initializeFromModel (energyMinimizerLoLBFGS.cpp:32-52): zero history
        const int launches = (M->m + kLbBlock - 1) / kLbBlock;
        if (int rc = M->bind(L, 2 * M->m + 1, LbLayout{M->m}.size(), (size_t)launches * kLbDots * kLbBlocks)) return rc;
        M->fresh = true;
        M->iterations = 0;
        M->cur = 0;
    }
    // at least one iteration per call (energyMinimizerLoLBFGS.cpp:199-201)
    if (int rc = begin_run(*M, L, f, false)) return rc;
    const int cur0 = M->cur, it0 = M->iterations;
    auto enq = [&](int iteration) {
        return L->precision == QM_FP64 ? lb_enqueue<double>(M, L, f, iteration, iteration == it0)
                                       : lb_enqueue<float>(M, L, f, iteration, iteration == it0);
    };
    int rc = drive(*M, L, enq);
    M->cur = (cur0 + (M->iterations - it0)) % M->m;
    // the next call's first direction: whatever computes forces on the lattice in
    // between, it starts from these
    HIP_TRY(hipMemcpyAsync(M->vecs[2 * M->m], static_cast<char*>(L->dSet[L->hCtrl.cur]) + 10 * (size_t)L->n * L->realSize,
                           5 * (size_t)L->n * L->realSize, hipMemcpyDeviceToDevice, L->stream));
    return rc;
}

int qm_lolbfgs_get_state(const qm_lolbfgs* m, int* iterations, double* forceMax) {
    if (!m) return fail(QM_EINVAL, "null minimizer");
    if (iterations) *iterations = m->iterations;
    if (forceMax) *forceMax = m->forceMax;
    return QM_OK;
}

}  // extern "C"

// ------------------------------------------------------------------ traces
template <typename M>
static int set_trace(M* m, int capacity) {
    if (!m || capacity < 0) return fail(QM_EINVAL, "bad argument");
    m->traceCap = capacity;
    m->trace.clear();
    return QM_OK;
}

template <typename M>
static int get_trace(const M* m, double* out, int cap, int* n) {
    if (!m || !n) return fail(QM_EINVAL, "bad argument");
    const int k = std::min<int>(cap, (int)m->trace.size());
    if (out && k > 0) std::memcpy(out, m->trace.data(), (size_t)k * sizeof(double));
    *n = k;
    return QM_OK;
}

extern "C" {
int qm_adam_set_trace(qm_adam* m, int capacity) { return set_trace(m, capacity); }
int qm_adam_get_trace(const qm_adam* m, double* forceMax, int cap, int* n) { return get_trace(m, forceMax, cap, n); }
int qm_nesterov_set_trace(qm_nesterov* m, int capacity) { return set_trace(m, capacity); }
int qm_nesterov_get_trace(const qm_nesterov* m, double* forceMax, int cap, int* n) {
    return get_trace(m, forceMax, cap, n);
}
int qm_lolbfgs_set_trace(qm_lolbfgs* m, int capacity) { return set_trace(m, capacity); }
int qm_lolbfgs_get_trace(const qm_lolbfgs* m, double* forceMax, int cap, int* n) {
    return get_trace(m, forceMax, cap, n);
}
}
