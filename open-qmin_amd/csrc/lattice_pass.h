// Device code shared by the lattice passes of the qmin HIP library (gfx950):
// the fused pass over halo-padded tiles (march_body) and the boundary pass
// (boundary_body), each compiled per pass mode (force only, FIRE, or the
// force with the Adam or Nesterov update) by the translation units that
// launch them.
#pragma once
#include "qmin_device.h"
#include "ldg_math.h"

namespace qmin {

#include "gen/ldg_stencils.inc"

__device__ __forceinline__ int wrapi(int v, int m) {
    v %= m;
    return v < 0 ? v + m : v;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block-wide sum of three doubles in a fixed order; result valid in thread 0.
template <int NT>
__device__ __forceinline__ void block_sum3(double& a, double& b, double& c, double (*red)[3]) {
    a = wave_sum(a);
    b = wave_sum(b);
    c = wave_sum(c);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) {
        red[w][0] = a;
        red[w][1] = b;
        red[w][2] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) {
            s0 += red[i][0];
            s1 += red[i][1];
            s2 += red[i][2];
        }
        a = s0;
        b = s1;
        c = s2;
    }
}

// Derivative at neighbour n along one transverse axis, with the reference's
// rules (landauDeGennesLCOtherForces.cpp:15-145): zero on objects, central on
// t == 0 or when neither side is an object, otherwise one-sided with an object
// above taking precedence.
template <typename R>
__device__ __forceinline__ void nbr_derivative(int tn, int tu, int td, const R* nq, const R* qu, const R* qd, R* out) {
    if (tn > 0) {
#pragma unroll
        for (int c = 0; c < 5; ++c) out[c] = R(0);
    } else if (tn == 0 || (td <= 0 && tu <= 0)) {
#pragma unroll
        for (int c = 0; c < 5; ++c) out[c] = R(0.5) * (qu[c] - qd[c]);
    } else if (tu > 0) {
#pragma unroll
        for (int c = 0; c < 5; ++c) out[c] = nq[c] - qd[c];
    } else {
#pragma unroll
        for (int c = 0; c < 5; ++c) out[c] = qu[c] - nq[c];
    }
}

// Raw force (phase - distortion) of a site whose neighbours all have central
// derivatives: the bulk L1..L4 forms composed with those differences into one
// linear 19-point operator (weights W), plus the quadratic L6 form.
// Uniform read-only data seen through the constant address space, so that the
// compiler fetches it with scalar loads.
template <typename R>
using ConstPtr = const R __attribute__((address_space(4)))*;

template <typename R, int TERMS, int HX, int HP>
__device__ __forceinline__ void fast_raw_force(const ForceConst& fc, ConstPtr<R> W, const R (*q)[5][HP],
                                               int sm, int sc, int sp, int h, const R* qc, R* F) {
#pragma unroll
    for (int c = 0; c < 5; ++c) F[c] = R(0);
    phase_force(R(fc.a), R(fc.b), R(fc.c), qc, F);
    R spatial[5] = {R(0), R(0), R(0), R(0), R(0)};
    if constexpr (TERMS == kOneConstant) {
#pragma unroll
        for (int c = 0; c < 5; ++c)
            spatial[c] = R(fc.L1) * (R(6) * qc[c] - q[sc][c][h - 1] - q[sc][c][h + 1] - q[sc][c][h - HX] -
                                     q[sc][c][h + HX] - q[sm][c][h] - q[sp][c][h]);
        l1_shape(spatial);
    } else if constexpr (TERMS == kMultiLinear) {
        ldg_fast_lin_a<HX, HP>(W, q, sm, sc, sp, h, spatial);
    } else if constexpr (TERMS == kMultiL4) {
        ldg_fast_lin_b<HX, HP>(W, q, sm, sc, sp, h, spatial);
    } else {
        R o6[5] = {R(0), R(0), R(0), R(0), R(0)};
        ldg_fast_lin_b_l6<HX, HP>(W, q, sm, sc, sp, h, qc, spatial, o6);
#pragma unroll
        for (int c = 0; c < 5; ++c) spatial[c] += R(fc.L6) * o6[c];
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) F[c] -= spatial[c];
}

// fv: the site's spatially varying field force, or null
template <typename R>
__device__ __forceinline__ void finish_bulk(const ForceConst& fc, R* F, const R* fv) {
    if (fc.semantics == 0) metric(F);
    if (fc.hasField) {
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] += R(fc.field[c]);
    }
    if (fv) {
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] += fv[c];
    }
    metric(F);
}

// Stores of the next state: not read again in this pass, so with NT they are
// streamed past L2 (non-temporal), which keeps L2 for the halo rows that
// neighbouring tiles read (nontemporal_stores has the rule).  A template
// parameter: of stores in the two branches of a flag, the compiler makes plain
// ones.
template <bool NT, typename R>
__device__ __forceinline__ void st_out(R* p, R v) {
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

template <bool NT, typename R>
__device__ __forceinline__ void st_site(R* field, long long n, long long i, const R* v) {
#pragma unroll
    for (int c = 0; c < 5; ++c) st_out<NT>(&field[c * n + i], v[c]);
}

// Coefficients of one Adam or Nesterov update, from the minimizer's device
// scalars as the previous iteration's finalize kernel left them.
template <typename R>
struct StepCoef {
    R b1, b1m1, b2, omb2, inv1, inv2, eps, mdt;  // Adam
    R dt, mu;                                     // Nesterov
};

template <typename R, int MODE>
__device__ __forceinline__ StepCoef<R> step_coef(const StepArgs& S) {
    StepCoef<R> k{};
    if constexpr (MODE == kAdamStep) {
        const double b1t = S.scal[0], b2t = S.scal[1];
        k.b1 = R(S.b1);
        k.b2 = R(S.b2);
        k.b1m1 = R(S.b1 - 1);
        k.omb2 = R(1 - S.b2);
        k.inv1 = R(1.0 / (1.0 - b1t));
        k.inv2 = R(1.0 / (1.0 - b2t));
        k.eps = R(S.eps);
        k.mdt = R(-S.dt);
    } else if constexpr (MODE == kNesterovStep) {
        // lambda and the scheduled momentum of this iteration
        // (energyMinimizerNesterovAG.cpp:101-108)
        const double oldLambda = S.scal[0];
        const double lambda = 0.5 * (1.0 + sqrt(1.0 + 4.0 * oldLambda * oldLambda));
        const double gamma = (1 - oldLambda) / lambda;
        k.mu = R(S.scheduled ? 1. + gamma : S.scal[1]);
        k.dt = R(S.dt);
    }
    return k;
}

// The minimizer's own entries of site i (Adam: m and s; Nesterov: the
// alternate sequence), loaded before the site's force is computed so that the
// force computation covers their latency.
template <typename R, int MODE>
__device__ __forceinline__ void step_load(const StepArgs& S, long long n, long long i, R (&pre)[2][5]) {
    const R* m = static_cast<const R*>(S.m);
#pragma unroll
    for (int c = 0; c < 5; ++c) pre[0][c] = m[c * n + i];
    if constexpr (MODE == kAdamStep) {
        const R* v = static_cast<const R*>(S.v);
#pragma unroll
        for (int c = 0; c < 5; ++c) pre[1][c] = v[c * n + i];
    }
}

// The update of component j (of site or lattice index j) from its q, force and
// entries (step_load): energyMinimizerAdam::adamStepCPU
// (energyMinimizerAdam.cpp:25-54; epsilon replaces sqrt(vc) where that is 0) or
// energyMinimizerNesterovAG::nesterovStepCPU (energyMinimizerNesterovAG.cpp:75-92).
// Stores the advanced entries (no other work-item reads them in the pass) and
// returns the new q.
template <typename R, int MODE, bool NT>
__device__ __forceinline__ R step_component(const StepArgs& S, const StepCoef<R>& k, long long j, R q, R F, R m0,
                                            R v0) {
    R* m = static_cast<R*>(S.m);
    if constexpr (MODE == kAdamStep) {
        R* v = static_cast<R*>(S.v);
        const R mm = k.b1 * m0 + k.b1m1 * F;
        const R vv = k.b2 * v0 + k.omb2 * (F * F);
        const R mc = mm * k.inv1;
        const R vc = vv * k.inv2;
        R root = sqrt(vc);
        if (root == R(0)) root = k.eps;
        st_out<NT>(&m[j], mm);
        st_out<NT>(&v[j], vv);
        return q + k.mdt * mc / root;
    } else {
        const R alt = q + k.dt * F;
        st_out<NT>(&m[j], alt);
        return alt + k.mu * (alt - m0);
    }
}

template <typename R, int MODE, bool NT>
__device__ __forceinline__ void step_site(const StepArgs& S, const StepCoef<R>& k, long long n, long long i,
                                          const R* q, const R* F, const R (&pre)[2][5], R* qn) {
#pragma unroll
    for (int c = 0; c < 5; ++c)
        qn[c] = step_component<R, MODE, NT>(S, k, c * n + i, q[c], F[c], pre[0][c],
                                            MODE == kAdamStep ? pre[1][c] : R(0));
}

// Sum of squares of the five stored components (the minimizers' |F|^2).
template <typename R>
__device__ __forceinline__ double sq5(const R* F) {
    double s = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c) s += double(F[c]) * double(F[c]);
    return s;
}

constexpr bool is_step_mode(int mode) { return mode == kAdamStep || mode == kNesterovStep; }

// Whether the fused pass loads the minimizer's entries before the site's force
// computation (their latency hidden behind it) or right before the update.
// Early loads keep 5 or 10 more values live across the force computation: in
// FP64 with L6 that costs a wave per SIMD (Adam 202 VGPRs against 146), and
// the late load is faster there (per iteration at 384^3: Adam 4.68 against
// 5.29 ms, Nesterov 3.51 against 4.33 ms); everywhere else the early load is
// (FP32 with L6: 2.30 against 2.51 and 1.85 against 2.02 ms; 256^3 with
// L1..L3: FP64 0.74 against 0.78 ms for Nesterov, FP32 0.56 against 0.59 ms
// for Adam).
template <typename R, int TERMS>
constexpr bool step_early_load() { return !(sizeof(R) == 8 && TERMS == kMultiL6); }

// FP32 force-only passes on the 512-thread tiles, without L6 (55-70 of 128
// registers): the next plane but one is loaded into registers before the force
// of the current one, and written to LDS a step later; each step waits for
// those loads before it stores its forces, so that the stores drain behind the
// next step's barrier instead of being waited for with the next plane's loads
// (vector memory operations complete in order on one counter).  At 256^3 a
// force computation (pass, boundary pass, synchronisation) takes 0.223 against
// 0.281 ms so; in FP64 (107 registers against 76) 0.369 against 0.365 ms, and
// FP64 keeps loading each plane at the top of its step.
template <typename R, int MODE, int TERMS, int TILE>
constexpr bool march_prefetch() {
    return sizeof(R) == 4 && MODE == kForce && TERMS != kMultiL6 && kTileThreads[TILE] == 512;
}

template <typename R>
__device__ __forceinline__ void wait_plane(const R (&a)[5], const R (&b)[5], int c) {
    asm volatile("" ::"v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(c) : "memory");
    asm volatile("" ::"v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(b[4]) : "memory");
}

// FIRE scalar step of energyMinimizerFIRE::fireStepCPU (energyMinimizerFIRE.cpp:77-145),
// run by one thread once all partial sums are in.
__device__ __forceinline__ void fire_scalar_step(Ctrl* ctrl, const FireConst& fp, double fnorm, double power, double vnorm,
                                 double* trace) {
    const int it = ctrl->iterations + 1;
    const double forceMax = sqrt(fnorm) / fp.nTotal;
    const double scaling = fnorm > 0. ? sqrt(vnorm / fnorm) : 0.0;
    double alpha = ctrl->alpha, dt = ctrl->dt;
    int nPos = ctrl->nPositive;
    ctrl->cKeep = 1.0 - alpha;
    ctrl->cForce = alpha * scaling;
    ctrl->identity = 0;
    if (power > 0 && it % 500 != 0) {
        if (nPos > fp.nMin) {
            dt = fmin(dt * fp.dtInc, fp.dtMax);
            alpha = alpha * fp.alphaDec;
            alpha = fmax(alpha, fp.alphaMin);
        }
        nPos += 1;
        ctrl->reset = 0;
    } else {
        nPos = 0;
        dt = dt * fp.dtDec;
        dt = fmax(dt, fp.dtMin);
        alpha = fp.alphaStart;
        ctrl->reset = 1;
    }
    ctrl->alpha = alpha;
    ctrl->dt = dt;
    ctrl->nPositive = nPos;
    ctrl->iterations = it;
    ctrl->forceMax = forceMax;
    ctrl->power = power;
    ctrl->fnorm = fnorm;
    ctrl->vnorm = vnorm;
    ctrl->scaling = scaling;
    if (trace && ctrl->traceLen < ctrl->traceCap) {
        double* t = trace + 6 * (long long)ctrl->traceLen;
        t[0] = forceMax;
        t[1] = power;
        t[2] = alpha;
        t[3] = dt;
        t[4] = scaling;
        t[5] = nPos;
        ctrl->traceLen += 1;
    }
    ctrl->cur ^= 1;
    if (isnan(forceMax)) ctrl->nanFlag = 1;
    ctrl->done = !(it < ctrl->maxIter && forceMax > fp.fc);
}

// This thread's share of the fixed-order sum of the partials of `total` slots.
__device__ __forceinline__ void fire_partials(const double* part, long long total, double& s0, double& s1, double& s2) {
    for (long long j = threadIdx.x; j < total; j += kReduceThreads) {
        s0 += part[3 * j + 0];
        s1 += part[3 * j + 1];
        s2 += part[3 * j + 2];
    }
}

// Velocity-Verlet drift and first half kick of one site with the pending FIRE
// velocity mix v = ck u + cf F, (1, 0) when none is pending and (0, 0) after a
// reset (energyMinimizerFIRE.cpp:117-144, velocityVerlet.cpp:8-40):
//   q + dt v + dt^2/2 F = q + (du u + df F),  v + dt/2 F = vu u + vf F.
// One rounding of q, and the products contracted by hand, so that the marching and
// the block passes round alike.  (The pass that keeps only Q and v drifts in a
// form of its own, fire_stream.hip, and rounds differently.)
template <typename R>
struct FireMove {
    R du, df, vu, vf, hdt;
};

template <typename R>
__device__ __forceinline__ FireMove<R> fire_move(const Ctrl* ctrl) {
    const double dt = ctrl->dt;
    const int reset = ctrl->reset, identity = ctrl->identity;
    const double ck = reset ? 0.0 : (identity ? 1.0 : ctrl->cKeep), cf = (reset || identity) ? 0.0 : ctrl->cForce;
    return {R(dt * ck), R(dt * cf + 0.5 * dt * dt), R(ck), R(cf + 0.5 * dt), R(0.5 * dt)};
}

template <typename R>
__device__ __forceinline__ R fire_drift(const FireMove<R>& m, R q, R u, R f) {
    return q + __builtin_elementwise_fma(m.du, u, m.df * f);
}

template <typename R>
__device__ __forceinline__ R fire_half_kick(const FireMove<R>& m, R u, R f) {
    return __builtin_elementwise_fma(m.vu, u, m.vf * f);
}

// One work-group's share of the fused pass: the column of tile `logical` (x
// tile fastest, then y tile, then z chunk) of the lattice described by A; its
// partial sums go to slot `slot`.
// NARROW: the tile is A.tw x A.th sites (an ensemble's lattices, whose rows may
// be shorter than TX), else TX x TY.  NT: non-temporal stores of the next state.
template <typename R, int MODE, int TERMS, int TILE, bool NARROW, bool NT>
__device__ __forceinline__ void march_body(const MarchArgs<R>& A, const int logical, const int slot) {
    using T = Tile<kTileTX[TILE], kTileTY[TILE], NARROW ? tile_rows<R>(TILE) : kTileTY[TILE]>;
    constexpr int kHX = T::HX, kHP = T::HP;
    __shared__ R sQ[3][5][kHP];
    __shared__ double sRed[T::Threads / 64][3];

    Ctrl* ctrl = A.ctrl;
    if ((MODE != kForce || A.gate) && ctrl->done) return;
    const int cur = ctrl->cur;
    const StateSet<R> in = A.set[cur];
    const StateSet<R> out = A.set[MODE == kForce ? cur : cur ^ 1];
    FireMove<R> mv{};
    if (MODE == kFire) mv = fire_move<R>(ctrl);
    StepCoef<R> sk{};
    if constexpr (is_step_mode(MODE)) sk = step_coef<R, MODE>(A.step);

    const int txi = logical % A.nbx;
    const int rest = logical / A.nbx;
    const int tyi = rest % A.nby;
    const int zc = rest / A.nby;
    const int z0 = zc * A.zchunk;
    const int z1 = min(z0 + A.zchunk, A.lz);

    const int lx = A.lx, ly = A.ly, lz = A.lz;
    const long long n = A.n;
    const long long plane = (long long)lx * ly;
    const int tid = threadIdx.x;
    const int tw = NARROW ? A.tw : T::TX, th = NARROW ? A.th : T::TY;
    const int ox = tid % tw, oy = tid / tw;
    const bool own = !NARROW || oy < th;   // a narrow tile may leave threads over
    const int x = txi * tw + ox, y = tyi * th + oy;
    const bool active = own && x < lx && y < ly;
    const int hOwn = own ? (oy + 1) * kHX + (ox + 1) : 0;
    const long long colOwn = own ? wrapi(x, lx) + (long long)lx * wrapi(y, ly) : 0;
    int hHalo = -1;
    long long colHalo = 0;
    if (tid < 2 * (tw + 2) + 2 * th) {
        const int k = tid, w = tw + 2;
        int hx, hy;
        if (k < 2 * w) {
            hx = k < w ? k : k - w;
            hy = k < w ? 0 : th + 1;
        } else {
            const int m = k - 2 * w;
            hx = m < th ? 0 : tw + 1;
            hy = 1 + (m < th ? m : m - th);
        }
        hHalo = hy * kHX + hx;
        colHalo = wrapi(txi * tw - 1 + hx, lx) + (long long)lx * wrapi(tyi * th - 1 + hy, ly);
    }

    // Stage plane z into slot s (FIRE: pending mix, drift and first half kick);
    // returns the owner's half-kicked velocity and class.  The own and the halo
    // site are loaded together in the FP32 passes that read Q alone (150^3 Adam:
    // 130 against 141 us per iteration); elsewhere that gains nothing (FIRE, FP32,
    // 256^3: 437 against 431 us; Nesterov, FP64, 192 x 150 x 130: 194 against 189).
    constexpr bool kTogether = sizeof(R) == 4 && MODE != kFire;
    auto load_site = [&](long long i, R* q, R* u, R* f) {
#pragma unroll
        for (int c = 0; c < 5; ++c) q[c] = in.q[c * n + i];
        if (MODE == kFire) {
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                u[c] = in.u[c * n + i];
                f[c] = in.f[c * n + i];
            }
        }
    };
    auto put_site = [&](int s, int h, R* q, const R* u, const R* f, R* vh) {
        if (MODE == kFire) {
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                q[c] = fire_drift(mv, q[c], u[c], f[c]);
                vh[c] = fire_half_kick(mv, u[c], f[c]);
            }
        }
#pragma unroll
        for (int c = 0; c < 5; ++c) sQ[s][c][h] = q[c];
    };
    auto stage = [&](int z, int s, R* vh, int& cOwn) {
        const long long zoff = plane * wrapi(z, lz);
        if constexpr (kTogether) {
            R q[5], hq[5];
            if (own) {
                cOwn = A.cls[colOwn + zoff];
                load_site(colOwn + zoff, q, nullptr, nullptr);
            }
            if (hHalo >= 0) load_site(colHalo + zoff, hq, nullptr, nullptr);
            if (own) put_site(s, hOwn, q, nullptr, nullptr, nullptr);
            if (hHalo >= 0) put_site(s, hHalo, hq, nullptr, nullptr, nullptr);
        } else {
            if (own) {
                R q[5], u[5], f[5];
                cOwn = A.cls[colOwn + zoff];
                load_site(colOwn + zoff, q, u, f);
                put_site(s, hOwn, q, u, f, vh);
            }
            if (hHalo >= 0) {
                R q[5], u[5], f[5], unused[5];
                load_site(colHalo + zoff, q, u, f);
                put_site(s, hHalo, q, u, f, unused);
            }
        }
    };

    constexpr bool kPF = march_prefetch<R, MODE, TERMS, TILE>();
    R pq[5], ph[5];   // kPF: Q of the next plane but one (own site, halo site) and the own class
    int pc = 0;
    auto fetch = [&](int z) {
        const long long zoff = plane * wrapi(z, lz);
        const long long i = colOwn + zoff;
        if (own) {
            pc = A.cls[i];
#pragma unroll
            for (int c = 0; c < 5; ++c) pq[c] = in.q[c * n + i];
        }
        if (hHalo >= 0) {
            const long long j = colHalo + zoff;
#pragma unroll
            for (int c = 0; c < 5; ++c) ph[c] = in.q[c * n + j];
        }
    };

    double pF = 0, pP = 0, pV = 0;
    R vhCur[5], vhNext[5];
    int cCur = 0, cNext = 0;
    stage(z0 - 1, 0, vhNext, cNext);
    stage(z0, 1, vhCur, cCur);
    if constexpr (kPF) {
        // waited for here, so that the loop's head waits for nothing
        fetch(z0 + 1);
        wait_plane(pq, ph, pc);
    }
    for (int z = z0; z < z1; ++z) {
        const int sm = (z - z0) % 3, sc = (z - z0 + 1) % 3, sp = (z - z0 + 2) % 3;
        if constexpr (kPF) {
            if (own) {
#pragma unroll
                for (int c = 0; c < 5; ++c) sQ[sp][c][hOwn] = pq[c];
            }
            if (hHalo >= 0) {
#pragma unroll
                for (int c = 0; c < 5; ++c) sQ[sp][c][hHalo] = ph[c];
            }
            cNext = pc;
            if (z + 1 < z1) fetch(z + 2);
        } else {
            stage(z + 1, sp, vhNext, cNext);
        }
        __syncthreads();
        R Fst[5];
        bool putF = false;
        if (active) {
            const long long i = colOwn + plane * z;
            R pre[2][5];
            if constexpr (is_step_mode(MODE) && step_early_load<R, TERMS>())
                if (cCur >= 0) step_load<R, MODE>(A.step, n, i, pre);
            R q[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) q[c] = sQ[sc][c][hOwn];
            if (cCur >= 0) {
                R F[5];
                if (cCur == 0) {
                    // re-opaque the weight pointer every step: the loads stay
                    // inside the loop instead of being hoisted and spilled
                    uint64_t wa = reinterpret_cast<uint64_t>(A.W);
                    asm volatile("" : "+s"(wa));
                    fast_raw_force<R, TERMS, kHX, kHP>(A.fc, reinterpret_cast<ConstPtr<R>>(wa), sQ, sm, sc, sp,
                                                       hOwn, q, F);
                    if (A.hvar) {
                        R fv[5];
                        varying_field_force(A.hvar, n, i, A.hvarP, fv);
                        finish_bulk(A.fc, F, fv);
                    } else {
                        finish_bulk<R>(A.fc, F, nullptr);
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < 5; ++c) F[c] = R(0);
                }
                if (MODE == kFire) {
                    R u[5];
#pragma unroll
                    for (int c = 0; c < 5; ++c) u[c] = __builtin_elementwise_fma(mv.hdt, F[c], vhCur[c]);
#pragma unroll
                    for (int c = 0; c < 5; ++c) {
                        st_out<NT>(&out.q[c * n + i], q[c]);
                        st_out<NT>(&out.u[c * n + i], u[c]);
                        st_out<NT>(&out.f[c * n + i], F[c]);
                    }
                    pF += qt_dot(F, F);
                    pP += qt_dot(F, u);
                    pV += qt_dot(u, u);
                } else if constexpr (is_step_mode(MODE)) {
                    R qn[5];
                    if constexpr (!step_early_load<R, TERMS>()) step_load<R, MODE>(A.step, n, i, pre);
                    step_site<R, MODE, NT>(A.step, sk, n, i, q, F, pre, qn);
                    st_site<NT>(out.q, n, i, qn);
                    if (A.storeF) st_site<NT>(out.f, n, i, F);
                    pF += sq5(F);
                } else if constexpr (kPF) {
#pragma unroll
                    for (int c = 0; c < 5; ++c) Fst[c] = F[c];
                    putF = true;
                } else {
#pragma unroll
                    for (int c = 0; c < 5; ++c) out.f[c * n + i] = F[c];
                }
            } else if (MODE == kFire) {
                // the boundary pass finishes U and F of this site
#pragma unroll
                for (int c = 0; c < 5; ++c) {
                    st_out<NT>(&out.q[c * n + i], q[c]);
                    st_out<NT>(&out.u[c * n + i], vhCur[c]);
                }
            }
        }
        if constexpr (kPF) {
            wait_plane(pq, ph, pc);
            if (putF) {
                const long long i = colOwn + plane * z;
#pragma unroll
                for (int c = 0; c < 5; ++c) out.f[c * n + i] = Fst[c];
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 5; ++c) vhCur[c] = vhNext[c];
        cCur = cNext;
    }
    if (MODE != kForce) {
        block_sum3<T::Threads>(pF, pP, pV, sRed);
        if (tid == 0) {
            A.partials[3 * (long long)slot + 0] = pF;
            A.partials[3 * (long long)slot + 1] = pP;
            A.partials[3 * (long long)slot + 2] = pV;
        }
    }
}

// The fused pass on a small lattice: a work-group owns a block of up to 16 x 4 x
// 4 sites, one thread per site, and stages the block with its one-site halo in
// LDS at once, so that a pass lasts one load latency and one force computation
// instead of marching through planes that each wait for their loads.  The halo
// is 1.5 sites per site, read mostly from L2.  FIRE iteration at 24^3, L1, FP64:
// 12 against 20 us, at 50^3, L1..L3: 21 against 28 us (three launches each;
// 8.7 and 18 us chained).
// CHAIN: a FIRE pass that takes the previous iteration's scalar step (ChainArgs).
template <typename R, int MODE, int TERMS, bool CHAIN>
__device__ __forceinline__ void block_body(const MarchArgs<R>& A, const int logical, const int slot) {
    using B = Block;
    constexpr int kHX = B::HX, kHP = B::HP;
    __shared__ R sQ[B::HZ][5][kHP];
    __shared__ double sRed[B::Threads / 64][3];

    static_assert(!CHAIN || MODE == kFire, "FIRE passes are chained");
    Ctrl* ctrl = A.ctrl;
    if (!CHAIN && (MODE != kForce || A.gate) && ctrl->done) return;
    const int cur = CHAIN ? A.chain.cur : ctrl->cur;
    const StateSet<R> in = A.set[cur];
    const StateSet<R> out = A.set[MODE == kForce ? cur : cur ^ 1];
    FireMove<R> mv{};
    if (MODE == kFire && !CHAIN) mv = fire_move<R>(ctrl);
    StepCoef<R> sk{};
    if constexpr (is_step_mode(MODE)) sk = step_coef<R, MODE>(A.step);

    const int lx = A.lx, ly = A.ly, lz = A.lz, tw = A.tw, th = A.th, td = A.zchunk;
    const long long n = A.n;
    const int x0 = logical % A.nbx * tw, y0 = logical / A.nbx % A.nby * th, z0 = logical / A.nbx / A.nby * td;
    const int tid = threadIdx.x;
    auto site = [&](int hx, int hy, int hz) {
        return wrapi(x0 - 1 + hx, lx) + (long long)lx * (wrapi(y0 - 1 + hy, ly) + (long long)ly * wrapi(z0 - 1 + hz, lz));
    };
    // the own site, then the halo: the planes below and above, the rims of the others
    const int ox = tid % tw, oy = tid / tw % th, oz = tid / tw / th;
    const bool own = oz < td, active = own && x0 + ox < lx && y0 + oy < ly && z0 + oz < lz;
    const long long i = own ? site(ox + 1, oy + 1, oz + 1) : 0;
    const int w = tw + 2, face = w * (th + 2), rim = 2 * w + 2 * th, halo = 2 * face + td * rim;
    constexpr int kRounds = (B::Halo + B::Threads - 1) / B::Threads;
    R q[5], u[5], f[5], hq[kRounds][5], hu[kRounds][5], hf[kRounds][5];
    int hAt[kRounds], hZ[kRounds];
    int cls = 1;
    auto load_site = [&](long long j, R* a, R* b, R* c) {
#pragma unroll
        for (int k = 0; k < 5; ++k) a[k] = in.q[k * n + j];
        if (MODE == kFire) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                b[k] = in.u[k * n + j];
                c[k] = in.f[k * n + j];
            }
        }
    };
    if (own) {
        cls = A.cls[i];
        load_site(i, q, u, f);
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int k = tid + r * B::Threads;
        hAt[r] = -1;
        if (k < halo) {
            int hx, hy, hz;
            if (k < 2 * face) {
                const int m = k < face ? k : k - face;
                hx = m % w;
                hy = m / w;
                hz = k < face ? 0 : td + 1;
            } else {
                const int m = (k - 2 * face) % rim;
                hz = 1 + (k - 2 * face) / rim;
                if (m < 2 * w) {
                    hx = m < w ? m : m - w;
                    hy = m < w ? 0 : th + 1;
                } else {
                    hx = m - 2 * w < th ? 0 : tw + 1;
                    hy = 1 + (m - 2 * w < th ? m - 2 * w : m - 2 * w - th);
                }
            }
            hAt[r] = hy * kHX + hx;
            hZ[r] = hz;
            load_site(site(hx, hy, hz), hq[r], hu[r], hf[r]);
        }
    }
    if constexpr (CHAIN) {
        // the previous iteration's scalar step, in every work-group while the
        // sites' loads are in flight; the first one keeps its outcome
        static_assert(B::Threads == kReduceThreads, "one work-group sums as fire_finalize_kernel does");
        __shared__ Ctrl sCtrl;
        double s0 = 0, s1 = 0, s2 = 0;
        if (A.chain.pending) {
            fire_partials(A.chain.prev, A.chain.total, s0, s1, s2);
            block_sum3<kReduceThreads>(s0, s1, s2, sRed);
        }
        if (tid == 0) {
            sCtrl = *ctrl;
            if (A.chain.pending && !sCtrl.done)
                fire_scalar_step(&sCtrl, A.chain.fire, s0, s1, s2, slot == 0 ? A.chain.trace : nullptr);
            if (slot == 0) *A.chain.next = sCtrl;
        }
        __syncthreads();
        if (sCtrl.done) return;
        mv = fire_move<R>(&sCtrl);
    }
    R pre[2][5];
    if constexpr (is_step_mode(MODE))
        if (active && cls >= 0) step_load<R, MODE>(A.step, n, i, pre);
    const int h = (oy + 1) * kHX + ox + 1;
    R vh[5];
    auto drift = [&](R* a, const R* b, const R* c, R* v2) {
        if (MODE == kFire) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                a[k] = fire_drift(mv, a[k], b[k], c[k]);
                if (v2) v2[k] = fire_half_kick(mv, b[k], c[k]);
            }
        }
    };
    if (own) {
        drift(q, u, f, vh);
#pragma unroll
        for (int k = 0; k < 5; ++k) sQ[oz + 1][k][h] = q[k];
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (hAt[r] >= 0) {
            drift(hq[r], hu[r], hf[r], nullptr);
#pragma unroll
            for (int k = 0; k < 5; ++k) sQ[hZ[r]][k][hAt[r]] = hq[r][k];
        }
    __syncthreads();
    double pF = 0, pP = 0, pV = 0;
    if (active && cls >= 0) {
        R F[5];
        if (cls == 0) {
            fast_raw_force<R, TERMS, kHX, kHP>(A.fc, reinterpret_cast<ConstPtr<R>>(reinterpret_cast<uint64_t>(A.W)), sQ,
                                               oz, oz + 1, oz + 2, h, q, F);
            if (A.hvar) {
                R fv[5];
                varying_field_force(A.hvar, n, i, A.hvarP, fv);
                finish_bulk(A.fc, F, fv);
            } else {
                finish_bulk<R>(A.fc, F, nullptr);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 5; ++k) F[k] = R(0);
        }
        if (MODE == kFire) {
#pragma unroll
            for (int k = 0; k < 5; ++k) vh[k] = __builtin_elementwise_fma(mv.hdt, F[k], vh[k]);
            pF = qt_dot(F, F);
            pP = qt_dot(F, vh);
            pV = qt_dot(vh, vh);
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                out.q[k * n + i] = q[k];
                out.u[k * n + i] = vh[k];
                out.f[k * n + i] = F[k];
            }
        } else if constexpr (is_step_mode(MODE)) {
            R qn[5];
            step_site<R, MODE, false>(A.step, sk, n, i, q, F, pre, qn);
            pF = sq5(F);
#pragma unroll
            for (int k = 0; k < 5; ++k) out.q[k * n + i] = qn[k];
            if (A.storeF) {
#pragma unroll
                for (int k = 0; k < 5; ++k) out.f[k * n + i] = F[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 5; ++k) out.f[k * n + i] = F[k];
        }
    } else if (MODE == kFire && active) {
        // the boundary pass finishes U and F of this site
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            out.q[k * n + i] = q[k];
            out.u[k * n + i] = vh[k];
        }
    }
    if (MODE != kForce) {
        block_sum3<B::Threads>(pF, pP, pV, sRed);
        if (tid == 0) {
            A.partials[3 * (long long)slot + 0] = pF;
            A.partials[3 * (long long)slot + 1] = pP;
            A.partials[3 * (long long)slot + 2] = pV;
        }
    }
}

// XCD-aware work-group order: consecutive hardware ids go round-robin over the
// 8 XCDs; each XCD gets a contiguous run of logical tiles, so that tiles sharing
// halos share an L2.  With PAIR, within each run of 64 tiles of an XCD its
// first 32 work-groups take the even tiles and the next 32 the odd ones, so
// that, if the XCD's 32 CUs receive its work-groups in order (two each),
// x-neighbouring tiles share a CU.  Measured at 256^3: 2.6% faster for the FP32
// 64x8 pass; 27% slower, with 64% more HBM reads, for the FP64 32x16 pass,
// which keeps the plain order.
template <bool PAIR>
__device__ __forceinline__ int xcd_logical(int b, int nb) {
    const int qb = nb >> 3, rb = nb & 7, xcd = b & 7;
    int j = b >> 3;
    if constexpr (PAIR) {
        const int per = qb + (xcd < rb ? 1 : 0);
        if (j < (per & ~63)) j = (j & ~63) + ((j & 31) << 1) + ((j >> 5) & 1);
    }
    return xcd * qb + min(xcd, rb) + j;
}

// Waves per SIMD asked of the compiler for the 256-thread tiles: four (at most
// 128 VGPRs) for the FP64 force-only pass with L6 on 32 x 8 (its tile by
// default), which needs 132 otherwise and
// spills 4 at 128, and is 2% faster so at 384^3 (2.68-2.69 against 2.74-2.77 ms);
// the Adam and Nesterov passes with L6 spill 18 and 11 registers at 128 and are
// slower (5.31 against 4.69 ms, 4.00 against 3.55 ms), so they and the rest keep
// what their registers give.
template <typename R, int MODE, int TERMS, int TILE>
constexpr int march_min_waves() {
    return (sizeof(R) == 8 && TERMS == kMultiL6 && MODE == kForce && TILE == kTile32x8) ? 4 : 1;
}

template <typename R, int MODE, int TERMS, int TILE, bool NT>
__global__ void __launch_bounds__(kTileThreads[TILE], (march_min_waves<R, MODE, TERMS, TILE>())) march_kernel(MarchArgs<R> A) {
    march_body<R, MODE, TERMS, TILE, false, NT>(A, xcd_logical<false>(blockIdx.x, A.nblocks), blockIdx.x);
}

// The 512-thread tiles (32 x 16, 64 x 8; 8 waves): two work-groups per CU need
// at least four waves per SIMD, i.e. at most 128 VGPRs.
template <typename R, int MODE, int TERMS, int TILE, bool NT>
__global__ void __launch_bounds__(kTileThreads[TILE], 4) march_wide_kernel(MarchArgs<R> A) {
    static_assert(kTileThreads[TILE] == 512, "512-thread tiles only");
    constexpr bool kPair = sizeof(R) == 4 && TILE == kTile64x8;
    march_body<R, MODE, TERMS, TILE, false, NT>(A, xcd_logical<kPair>(blockIdx.x, A.nblocks), blockIdx.x);
}

// Waves per SIMD asked of the compiler for the block pass: left alone it holds
// the operands of a whole stencil in registers (213 to 256 in FP64, one or two
// waves); at four, 52 to 122 do without spills, at three 134 with FP64 L6 and 132
// to 149 in a chained FP64 pass.
template <typename R, int TERMS, bool CHAIN>
constexpr int block_min_waves() {
    return sizeof(R) == 4 ? 4 : (TERMS == kMultiL6 ? 2 : (CHAIN ? 3 : 4));
}

template <typename R, int MODE, int TERMS, bool CHAIN>
__global__ void __launch_bounds__(Block::Threads, (block_min_waves<R, TERMS, CHAIN>())) block_kernel(MarchArgs<R> A) {
    block_body<R, MODE, TERMS, CHAIN>(A, xcd_logical<false>(blockIdx.x, A.nblocks), blockIdx.x);
}

// The pass of one lattice with tile `tile` (a halo-padded one, or kBlock).
template <typename R, int MODE, int TERMS, bool NT>
const void* march_fn_tile(int tile) {
    switch (tile) {
        case kTile64x4: return reinterpret_cast<const void*>(&march_kernel<R, MODE, TERMS, kTile64x4, NT>);
        case kTile32x16: return reinterpret_cast<const void*>(&march_wide_kernel<R, MODE, TERMS, kTile32x16, NT>);
        case kTile64x8: return reinterpret_cast<const void*>(&march_wide_kernel<R, MODE, TERMS, kTile64x8, NT>);
        case kBlock: return reinterpret_cast<const void*>(&block_kernel<R, MODE, TERMS, false>);
        default: return reinterpret_cast<const void*>(&march_kernel<R, MODE, TERMS, kTile32x8, NT>);
    }
}

template <typename R, int MODE, bool NT>
const void* march_fn_terms(int terms, int tile) {
    switch (terms) {
        case kOneConstant: return march_fn_tile<R, MODE, kOneConstant, NT>(tile);
        case kMultiLinear: return march_fn_tile<R, MODE, kMultiLinear, NT>(tile);
        case kMultiL4: return march_fn_tile<R, MODE, kMultiL4, NT>(tile);
        default: return march_fn_tile<R, MODE, kMultiL6, NT>(tile);
    }
}

// (force passes store F plainly)
template <typename R, int MODE>
const void* march_fn_mode(int terms, int tile, bool nt) {
    if constexpr (MODE == kForce)
        return march_fn_terms<R, MODE, false>(terms, tile);
    else
        return nt ? march_fn_terms<R, MODE, true>(terms, tile) : march_fn_terms<R, MODE, false>(terms, tile);
}

// The fused pass over many lattices in one launch: map[b] = {lattice, logical
// tile} for hardware work-group b, laid out by the host in XCD-aware order.
template <typename R, int MODE, int TERMS, int TILE>
__global__ void __launch_bounds__(kTileThreads[TILE]) march_batch_kernel(const MarchArgs<R>* __restrict__ descs,
                                                               const int2* __restrict__ map) {
    // uniform over the work-group: read once, keep in scalar registers
    const int lat = __builtin_amdgcn_readfirstlane(map[blockIdx.x].x);
    const int logical = __builtin_amdgcn_readfirstlane(map[blockIdx.x].y);
    march_body<R, MODE, TERMS, TILE, true, true>(descs[lat], logical, logical);
}

template <typename R, int MODE, int TERMS, int TILE>
__global__ void __launch_bounds__(kTileThreads[TILE], 4) march_wide_batch_kernel(
    const MarchArgs<R>* __restrict__ descs, const int2* __restrict__ map) {
    static_assert(kTileThreads[TILE] == 512, "512-thread tiles only");
    const int lat = __builtin_amdgcn_readfirstlane(map[blockIdx.x].x);
    const int logical = __builtin_amdgcn_readfirstlane(map[blockIdx.x].y);
    march_body<R, MODE, TERMS, TILE, true, true>(descs[lat], logical, logical);
}

// ---------------------------------------------------------------- boundary pass

template <typename R>
__device__ __forceinline__ void gload(const R* base, long long n, long long i, R* v) {
#pragma unroll
    for (int c = 0; c < 5; ++c) v[c] = base[c * n + i];
}

// Work-group `blk` of the boundary pass of the lattice described by A, one lane
// per site: the stencils of many sites (boundary_lanes has the rule).
template <typename R, int MODE, int TERMS>
__device__ __forceinline__ void boundary_site_body(const BoundaryArgs<R>& A, const int blk) {
    __shared__ double sRed[kBoundaryThreads / 64][3];
    Ctrl* ctrl = A.ctrl;
    if ((MODE != kForce || A.gate) && ctrl->done) return;
    const int cur = ctrl->cur;
    // FIRE: the drifted state the fused pass has written; otherwise the current one
    const StateSet<R> st = A.set[MODE == kFire ? cur ^ 1 : cur];
    const R hdt = MODE == kFire ? R(0.5 * ctrl->dt) : R(0);
    StepCoef<R> sk{};
    if constexpr (is_step_mode(MODE)) sk = step_coef<R, MODE>(A.step);
    const long long n = A.n;
    const int lx = A.lx, ly = A.ly, lz = A.lz;
    double pF = 0, pP = 0, pV = 0;

    const long long k = (long long)blk * kBoundaryThreads + threadIdx.x;
    if (k < A.nsites) {
        const long long i = A.sites[k];
        R pre[2][5];
        if constexpr (is_step_mode(MODE)) step_load<R, MODE>(A.step, n, i, pre);
        const int self = A.types[i];
        const int x = int(i % lx), y = int((i / lx) % ly), z = int(i / ((long long)lx * ly));
        // neighbour sites in the reference order xd, xu, yd, yu, zd, zu
        long long nbi[6];
        nbi[0] = wrapi(x - 1, lx) + (long long)lx * (y + (long long)ly * z);
        nbi[1] = wrapi(x + 1, lx) + (long long)lx * (y + (long long)ly * z);
        nbi[2] = x + (long long)lx * (wrapi(y - 1, ly) + (long long)ly * z);
        nbi[3] = x + (long long)lx * (wrapi(y + 1, ly) + (long long)ly * z);
        nbi[4] = x + (long long)lx * (y + (long long)ly * wrapi(z - 1, lz));
        nbi[5] = x + (long long)lx * (y + (long long)ly * wrapi(z + 1, lz));
        R xin[125];
        int tn[6];
        gload(st.q, n, i, xin);
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            tn[d] = A.types[nbi[d]];
            gload(st.q, n, nbi[d], xin + 5 + 5 * d);
        }
        // transverse derivatives of each neighbour (along-axis entries are unused)
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            const int axis = d / 2;
            const int nx = d == 0 ? wrapi(x - 1, lx) : (d == 1 ? wrapi(x + 1, lx) : x);
            const int ny = d == 2 ? wrapi(y - 1, ly) : (d == 3 ? wrapi(y + 1, ly) : y);
            const int nz = d == 4 ? wrapi(z - 1, lz) : (d == 5 ? wrapi(z + 1, lz) : z);
#pragma unroll
            for (int ax = 0; ax < 3; ++ax) {
                R* out = xin + 35 + 15 * d + 5 * ax;
                if (ax == axis) {
#pragma unroll
                    for (int c = 0; c < 5; ++c) out[c] = R(0);
                    continue;
                }
                const long long iu = ax == 0 ? wrapi(nx + 1, lx) + (long long)lx * (ny + (long long)ly * nz)
                                   : ax == 1 ? nx + (long long)lx * (wrapi(ny + 1, ly) + (long long)ly * nz)
                                             : nx + (long long)lx * (ny + (long long)ly * wrapi(nz + 1, lz));
                const long long idn = ax == 0 ? wrapi(nx - 1, lx) + (long long)lx * (ny + (long long)ly * nz)
                                    : ax == 1 ? nx + (long long)lx * (wrapi(ny - 1, ly) + (long long)ly * nz)
                                              : nx + (long long)lx * (ny + (long long)ly * wrapi(nz - 1, lz));
                R qu[5], qd[5];
                gload(st.q, n, iu, qu);
                gload(st.q, n, idn, qd);
                nbr_derivative(tn[d], int(A.types[iu]), int(A.types[idn]), xin + 5 + 5 * d, qu, qd, out);
            }
        }
        const R* q = xin;
        R F[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] = R(0);
        phase_force(R(A.fc.a), R(A.fc.b), R(A.fc.c), q, F);
        R spatial[5];
        if (self == -1) {
            // boundaryL1Force: only object-facing directions (lcForces.h:39-63)
#pragma unroll
            for (int c = 0; c < 5; ++c) spatial[c] = R(0);
#pragma unroll
            for (int d = 0; d < 6; ++d)
                if (tn[d] > 0) {
                    const R* opp = xin + 5 + 5 * (d ^ 1);
#pragma unroll
                    for (int c = 0; c < 5; ++c) spatial[c] -= (opp[c] - q[c]);
                }
#pragma unroll
            for (int c = 0; c < 5; ++c) spatial[c] *= R(A.fc.L1);
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                R lap = R(6) * q[c];
#pragma unroll
                for (int d = 0; d < 6; ++d) lap -= xin[5 + 5 * d + c];
                spatial[c] = R(A.fc.L1) * lap;
            }
        }
        l1_shape(spatial);
        if constexpr (TERMS != kOneConstant) {
            R acc[3][5];
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int c = 0; c < 5; ++c) acc[t][c] = R(0);
            int bcase = 0;
            if (self == -1) {
                int xx = 0, yy = 0, zz = 0;
                if (tn[1] > 0) xx = 1;
                if (tn[0] > 0) xx = 2;
                if (tn[3] > 0) yy = 1;
                if (tn[2] > 0) yy = 2;
                if (tn[5] > 0) zz = 1;
                if (tn[4] > 0) zz = 2;
                bcase = xx + 4 * yy + 16 * zz;
            }
            ldg_boundary_lin(bcase, xin, acc);
#pragma unroll
            for (int c = 0; c < 5; ++c) spatial[c] += R(A.fc.L2) * acc[0][c];
#pragma unroll
            for (int c = 0; c < 5; ++c) spatial[c] += R(A.fc.L3) * acc[1][c];
#pragma unroll
            for (int c = 0; c < 5; ++c) spatial[c] += R(A.fc.L4) * acc[2][c];
            if constexpr (TERMS == kMultiL6) {
                R o6[5];
                ldg_boundary_l6(bcase, xin, o6);
#pragma unroll
                for (int c = 0; c < 5; ++c) spatial[c] += R(A.fc.L6) * o6[c];
            }
        }
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] -= spatial[c];
        R fv[5];
        if (A.hvar) varying_field_force(A.hvar, n, i, A.hvarP, fv);
        if (self == 0) {
            // a bulk site with a one-sided neighbour derivative: bulk semantics
            finish_bulk(A.fc, F, A.hvar ? fv : nullptr);
        } else {
#pragma unroll
            for (int d = 0; d < 6; ++d)
                if (tn[d] > 0) add_anchoring_force(A.objects[tn[d] - 1], q, xin + 5 + 5 * d, F);
            if (A.fc.hasField) {
#pragma unroll
                for (int c = 0; c < 5; ++c) F[c] += R(A.fc.field[c]);
            }
            if (A.hvar) {
#pragma unroll
                for (int c = 0; c < 5; ++c) F[c] += fv[c];
            }
            metric(F);
        }
        if (MODE == kFire) {
            R u[5];
            gload(st.u, n, i, u);
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                u[c] = u[c] + hdt * F[c];
                st.u[c * n + i] = u[c];
                st.f[c * n + i] = F[c];
            }
            pF = qt_dot(F, F);
            pP = qt_dot(F, u);
            pV = qt_dot(u, u);
        } else if constexpr (is_step_mode(MODE)) {
            const StateSet<R> out = A.set[cur ^ 1];
            R qn[5];
            step_site<R, MODE, false>(A.step, sk, n, i, q, F, pre, qn);
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                out.q[c * n + i] = qn[c];
                out.f[c * n + i] = F[c];
            }
            pF = sq5(F);
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) st.f[c * n + i] = F[c];
        }
    }
    if (MODE == kForce) return;
    block_sum3<kBoundaryThreads>(pF, pP, pV, sRed);
    if (threadIdx.x == 0) {
        const long long slot = A.marchBlocks + blk;
        A.partials[3 * slot + 0] = pF;
        A.partials[3 * slot + 1] = pP;
        A.partials[3 * slot + 2] = pV;
    }
}

// The same for few sites: eight lanes evaluate one site.  Lane d < 6 loads the neighbour in direction d (x-,
// x+, y-, y+, z-, z+) and the four sites beside it that its transverse
// derivatives need, takes its share of the L1 term and, if the neighbour is an
// object, the anchoring on it; then all lanes take turns at the terms of the
// site's stencil, whose inputs the six have put in LDS, and their sums are added.
//
// The pass is bound by the length of one wave's path, not by throughput: one
// lane per site loaded 155 values and ran through up to 27 straight-line
// stencils (80 KB of code in FP64).  50^3 with walls and a sphere, L1..L3, FP64:
// 8 against 24 us; four spheres with L1..L6 17 against 54 us.
template <typename R, int MODE, int TERMS>
__device__ __forceinline__ void boundary_lanes_body(const BoundaryArgs<R>& A, const int blk) {
    constexpr bool kMulti = TERMS != kOneConstant;
    constexpr int kOne = 125, kRow = kMulti ? 127 : 1;   // inputs of a site in LDS, odd row length
    __shared__ R sx[kBoundaryGroup][kRow];
    __shared__ double sRed[kBoundaryThreads / 64][3];
    Ctrl* ctrl = A.ctrl;
    if ((MODE != kForce || A.gate) && ctrl->done) return;
    const int cur = ctrl->cur;
    // FIRE: the drifted state the fused pass has written; otherwise the current one
    const StateSet<R> st = A.set[MODE == kFire ? cur ^ 1 : cur];
    const R hdt = MODE == kFire ? R(0.5 * ctrl->dt) : R(0);
    StepCoef<R> sk{};
    if constexpr (is_step_mode(MODE)) sk = step_coef<R, MODE>(A.step);
    const long long n = A.n;
    const int lx = A.lx, ly = A.ly, lz = A.lz;
    // a wave takes eight consecutive entries of the site list, whose lanes of one
    // direction are neighbours: where the sites are, their loads share lines
    constexpr int kPer = 64 / kBoundaryLanes;
    const int d = (threadIdx.x & 63) / kPer, g = (threadIdx.x >> 6) * kPer + threadIdx.x % kPer;
    const int axis = d >> 1;
    // index offset to the next site up or down an axis of m sites from coordinate v
    auto step = [](int v, int m, int stride, bool up) {
        return up ? (v == m - 1 ? -(m - 1) * stride : stride) : (v == 0 ? (m - 1) * stride : -stride);
    };
    double pF = 0, pP = 0, pV = 0;

    {
        const long long k = (long long)blk * kBoundaryGroup + g;
        const bool have = k < A.nsites;
        const int i = A.sites[have ? k : A.nsites - 1];   // site indices fit 31 bits
        const int self = A.types[i];
        const unsigned row = unsigned(i) / unsigned(lx);
        const int x = i - int(row) * lx, z = int(row / unsigned(ly)), y = int(row) - z * ly;
        // the entries that lane d < 5 finishes component d with
        const long long own = (d < 5 ? d : 0) * n + i;
        R pre0 = R(0), pre1 = R(0);
        if constexpr (MODE == kFire) pre0 = st.u[own];
        if constexpr (is_step_mode(MODE)) pre0 = static_cast<const R*>(A.step.m)[own];
        if constexpr (MODE == kAdamStep) pre1 = static_cast<const R*>(A.step.v)[own];
        R q[5], nq[5];
        gload(st.q, n, i, q);
        int tn = 0;
        if (d < 6) {
            // coordinate, length and stride of the neighbour's axis and of the two others
            const int v0 = axis == 0 ? x : (axis == 1 ? y : z), m0 = axis == 0 ? lx : (axis == 1 ? ly : lz);
            const int plane = lx * ly;
            const int nb = i + step(v0, m0, axis == 0 ? 1 : (axis == 1 ? lx : plane), d & 1);
            tn = A.types[nb];
            gload(st.q, n, nb, nq);
            if constexpr (kMulti) {
                int tu[2], td[2];
                R qu[2][5], qd[2][5];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int ax = axis + 1 + t >= 3 ? axis - 2 + t : axis + 1 + t;
                    const int v = ax == 0 ? x : (ax == 1 ? y : z), m = ax == 0 ? lx : (ax == 1 ? ly : lz),
                              stride = ax == 0 ? 1 : (ax == 1 ? lx : plane);
                    const int iu = nb + step(v, m, stride, true), id = nb + step(v, m, stride, false);
                    tu[t] = A.types[iu];
                    td[t] = A.types[id];
                    gload(st.q, n, iu, qu[t]);
                    gload(st.q, n, id, qd[t]);
                }
#pragma unroll
                for (int c = 0; c < 5; ++c) sx[g][5 + 5 * d + c] = nq[c];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int ax = axis + 1 + t >= 3 ? axis - 2 + t : axis + 1 + t;
                    R out[5];
                    nbr_derivative(tn, tu[t], td[t], nq, qu[t], qd[t], out);
#pragma unroll
                    for (int c = 0; c < 5; ++c) sx[g][35 + 15 * d + 5 * ax + c] = out[c];
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) nq[c] = q[c];
            if constexpr (kMulti) {
                if (d == 6) {
#pragma unroll
                    for (int c = 0; c < 5; ++c) sx[g][c] = q[c];
                } else {
                    sx[g][kOne] = R(1);
                }
            }
        }
        // which neighbours are objects, bit d per direction
        const unsigned long long facing = __ballot(d < 6 && tn > 0) >> (threadIdx.x % kPer);
        unsigned faces = 0;
#pragma unroll
        for (int k = 0; k < 6; ++k) faces |= unsigned(facing >> (kPer * k) & 1) << k;
        // this lane's share of what is added to the phase force.  L1: the bulk
        // Laplacian, or next to an object (boundaryL1Force, lcForces.h:39-63) only
        // the neighbours opposite to one
        R P[5];
        const bool l1 = d < 6 && (self == -1 ? (faces >> (d ^ 1)) & 1 : true);
#pragma unroll
        for (int c = 0; c < 5; ++c) P[c] = l1 ? R(A.fc.L1) * (nq[c] - q[c]) : R(0);
        l1_shape(P);
        if (self == -1 && tn > 0) add_anchoring_force(A.objects[tn - 1], q, nq, P);
        if constexpr (kMulti) {
            // boundary case: an object above (1) or below (2, taking precedence) on
            // each axis (lcForces.h:13-25)
            const int ox = (faces & 1) ? 2 : (faces >> 1) & 1, oy = (faces & 4) ? 2 : (faces >> 3) & 1,
                      oz = (faces & 16) ? 2 : (faces >> 5) & 1;
            const int bcase = self == -1 ? ox + 3 * oy + 9 * oz : 0;
            __syncthreads();
            auto terms = [&](const BoundaryTerm<R>* t, int rounds) {
                t += bcase * 5 * rounds * kBoundaryLanes + d;
#pragma unroll 4
                for (int r = 0; r < rounds; ++r)
#pragma unroll
                    for (int c = 0; c < 5; ++c) {
                        const BoundaryTerm<R> e = t[(c * rounds + r) * kBoundaryLanes];
                        P[c] -= e.coef * (sx[g][e.ab & 255] * sx[g][e.ab >> 8]);
                    }
            };
            terms(A.terms, kBoundaryLinRounds);
            if constexpr (TERMS == kMultiL6)
                terms(A.terms + kBoundaryCases * 5 * kBoundaryLinRounds * kBoundaryLanes, kBoundaryQuadRounds);
            __syncthreads();
        }
#pragma unroll
        for (int o = kPer; o < 64; o <<= 1)
#pragma unroll
            for (int c = 0; c < 5; ++c) P[c] += __shfl_xor(P[c], o, 64);
        R F[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] = R(0);
        phase_force(R(A.fc.a), R(A.fc.b), R(A.fc.c), q, F);
#pragma unroll
        for (int c = 0; c < 5; ++c) F[c] += P[c];
        R fv[5] = {R(0), R(0), R(0), R(0), R(0)};
        if (A.hvar) varying_field_force(A.hvar, n, i, A.hvarP, fv);
        // a bulk site with a one-sided neighbour derivative has bulk semantics
        if (self == 0 && A.fc.semantics == 0) metric(F);
        if (A.fc.hasField) {
#pragma unroll
            for (int c = 0; c < 5; ++c) F[c] += R(A.fc.field[c]);
        }
        if (A.hvar) {
#pragma unroll
            for (int c = 0; c < 5; ++c) F[c] += fv[c];
        }
        metric(F);
        R Fd = F[0], qd = q[0];
#pragma unroll
        for (int c = 1; c < 5; ++c) {
            Fd = d == c ? F[c] : Fd;
            qd = d == c ? q[c] : qd;
        }
        const bool put = have && d < 5;
        if (MODE == kFire) {
            const R ud = pre0 + hdt * Fd;
            const R u0 = __shfl(ud, threadIdx.x % kPer, 64);   // component 0's, for the QT products' F_0 u_3 and u_0 u_3
            if (put) {
                st.u[own] = ud;
                st.f[own] = Fd;
                const double f = double(Fd), u = double(ud);
                pF += f * f + (d == 3 ? double(F[0]) * f : 0.0);
                pP += f * u + (d == 3 ? double(F[0]) * u : 0.0);
                pV += u * u + (d == 3 ? double(u0) * u : 0.0);
            }
        } else if constexpr (is_step_mode(MODE)) {
            if (put) {
                const StateSet<R> out = A.set[cur ^ 1];
                out.q[own] = step_component<R, MODE, false>(A.step, sk, own, qd, Fd, pre0, pre1);
                out.f[own] = Fd;
                pF += double(Fd) * double(Fd);
            }
        } else {
            if (put) st.f[own] = Fd;
        }
    }
    if (MODE == kForce) return;
    block_sum3<kBoundaryThreads>(pF, pP, pV, sRed);
    if (threadIdx.x == 0) {
        const long long slot = A.marchBlocks + blk;
        A.partials[3 * slot + 0] = pF;
        A.partials[3 * slot + 1] = pP;
        A.partials[3 * slot + 2] = pV;
    }
}

template <typename R, int MODE, int TERMS, bool LANES>
__device__ __forceinline__ void boundary_body(const BoundaryArgs<R>& A, const int blk) {
    if constexpr (LANES)
        boundary_lanes_body<R, MODE, TERMS>(A, blk);
    else
        boundary_site_body<R, MODE, TERMS>(A, blk);
}

template <typename R, int MODE, int TERMS, bool LANES>
__global__ void __launch_bounds__(kBoundaryThreads) boundary_kernel(BoundaryArgs<R> A) {
    boundary_body<R, MODE, TERMS, LANES>(A, blockIdx.x);
}

template <typename R, int MODE, int TERMS, bool LANES>
__global__ void __launch_bounds__(kBoundaryThreads) boundary_batch_kernel(
    const BoundaryArgs<R>* __restrict__ descs, const int2* __restrict__ map) {
    const int lat = __builtin_amdgcn_readfirstlane(map[blockIdx.x].x);
    const int blk = __builtin_amdgcn_readfirstlane(map[blockIdx.x].y);
    boundary_body<R, MODE, TERMS, LANES>(descs[lat], blk);
}

// The kernels of a force's stencil variant; neither form distinguishes L1..L3
// from L1..L4.
template <typename R, int MODE>
const void* boundary_fn(int terms, bool lanes) {
    if (terms == kOneConstant)
        return lanes ? reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kOneConstant, true>)
                     : reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kOneConstant, false>);
    if (terms == kMultiL6)
        return lanes ? reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kMultiL6, true>)
                     : reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kMultiL6, false>);
    return lanes ? reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kMultiLinear, true>)
                 : reinterpret_cast<const void*>(&boundary_kernel<R, MODE, kMultiLinear, false>);
}

}  // namespace qmin
