// Learned warm start: a small fully-convolutional 3-D network maps a lattice's
// geometry (site types, anchoring tensors and strengths, a chosen far-field
// director) to an initial Q field, from which FIRE then minimizes.  Random-start
// FIRE stays the fallback and decides the final state.
//
// Kernels (BF16 operands on the matrix cores, FP32 accumulation):
//  * conv_fwd_kernel: 3x3x3 dilated periodic convolution as an implicit GEMM,
//    D[site][cout] = sum_{tap, cin} X[site + dil*tap][cin] Wt[tap][cout][cin],
//    on the matrix cores: a wave owns 64 consecutive sites and all output
//    channels; with 64 input channels each lane feeds 8 consecutive input
//    channels of one neighbour site to v_mfma_f32_16x16x32_bf16 (activations
//    are channels-last, so that is one 16-byte load), with 16 or 32 input
//    channels 4 of them to v_mfma_f32_16x16x16_bf16; the tap's weights come
//    from LDS.
//    Optional ReLU on the input as it is read, bias, and an output mask (the
//    ReLU derivative of the previous layer when the kernel runs backwards).
//  * The input gradient is the same kernel with the taps mirrored and the
//    weights transposed (Wbd[26 - tap][cin][cout] = Wt[tap][cout][cin]).
//  * conv_wgrad_kernel: dWt[tap][cout][cin] = sum_site G[site][cout]
//    X[site + dil*tap][cin], a GEMM over sites per (tap, slot of sites); the
//    slots' partial sums are added in a fixed order by wgrad_reduce_kernel.
//  * Elementwise kernels: features, loss gradient, bias gradient, Adam with the
//    BF16 (and mirrored) weight copies, writing the prediction into a lattice.
#include <algorithm>
#include <cstdint>

#include "qmin_internal.h"

namespace qmin {
namespace ws {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// BF16 pairs with the sign bit set (negative values and -0) -> +0
__device__ __forceinline__ unsigned relu2(unsigned w) {
    typedef short v2s __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(v2s, w), v2s{0, 0}));
}

constexpr int kTaps = 27;
constexpr int kWsThreads = 256;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

// round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

__device__ __forceinline__ int wrapd(int v, int m) {
    v %= m;
    return v < 0 ? v + m : v;
}

__device__ __forceinline__ long long tap_site(int x, int y, int z, int tap, int dil, int lx, int ly, int lz) {
    const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
    return wrapd(x + dil * dx, lx) + (long long)lx * (wrapd(y + dil * dy, ly) + (long long)ly * wrapd(z + dil * dz, lz));
}

// One tile of the forward kernel: `rows` consecutive lattice rows (y fastest),
// of each a segment of w sites, as the host chose it (choose_conv_tile).
struct ConvTile {
    int w, nseg;    // segment length along x, segments per row
    int rows;       // rows per work-group
    int halo;       // sites staged on each side of a segment: dil, or 0
    int fold;       // 1: a step stages the rows of one (dy, dz) for its three taps; 0: the sites of one tap
    // order of the row groups: blocks of `block` consecutive groups, and within
    // a block the groups dil planes apart (stride groups) one after the other,
    // so that the planes z - dil, z and z + dil are found in L2
    int groups, stride, turns, block;
};

struct ConvArgs {
    const uint16_t* x;     // [n][cin] bf16
    const uint16_t* wt;    // [27][cout][cin] bf16
    const float* bias;     // [cout] or null
    const uint16_t* mask;  // [n][cout] bf16: output zeroed where mask <= 0 (null: none)
    uint16_t* ybf;         // [n][cout] bf16 output, or
    float* yf;             // [n][cout] fp32 output
    long long n;
    int cin, cout, lx, ly, lz, dil, reluIn;
    ConvTile tile;
    int nblocks;
    int vecX, vecW, vecOut;   // x, wt, and ybf with mask are 16-byte aligned (else x at 32 or fewer channels and
                              // wt take 8-byte loads, and ybf element stores)
};

constexpr int kFwdMT = 4;                                     // 16-site row tiles per wave in the forward kernel
constexpr int kFwdSites = kWsThreads / 64 * 16 * kFwdMT;      // sites a work-group computes
constexpr int kFwdSlots = 288;                                // sites it stages per step at most
constexpr int kFwdRows = 32;                                  // rows it covers at most
constexpr int kFwdBlock = 16;                                 // row groups taken together along z at most

// 3x3x3 dilated periodic convolution as an implicit GEMM.  A work-group owns up
// to 256 sites of whole row segments, each wave 64 of them and all output
// channels.  For each (dy, dz) it stages the segments' neighbour rows in LDS
// once, ReLU applied, with the weights of the three taps that differ in dx
// only: these read the same rows at three offsets.  The next step's rows and
// weights are loaded into registers while the matrix instructions of the
// current one run.  Rows in LDS are padded (8 BF16 at 64 channels, 4 below), so
// that the 16 sites of a fragment fall on different banks.
//
// Bound by latency: with two work-groups per CU (72.7 KB of LDS each at 64
// channels) the waves wait half of their time on operand reads and on the two
// barriers of a step, while LDS is busy 40% of the clocks (bank conflicts 14%),
// the matrix cores 28%, the vector units 26% and the L1 18% (64 -> 64, 128^3).
// Gathering every tap's operand from L2 instead, 27 reads of each site, left the
// kernel waiting on those gathers.  At 128^3, before and now: 64 -> 64 channels 1.46
// and 0.65 ms (710 TFLOP/s), 64 -> 16 0.99 and 0.36, 32 -> 64 0.78 and 0.45,
// 16 -> 32 0.43 and 0.13 ms.  Measured and not kept: 320 slots, with which the
// 64 -> 16 kernel has two work-groups per CU instead of three (0.52 ms); three
// waves per SIMD at 32 channels (0.54 ms: spills); the loads after the first tap
// and a raised wave priority during the taps (no difference).
template <int NT, int KT>
__global__ void __launch_bounds__(kWsThreads, 2) conv_fwd_kernel(ConvArgs a) {
    // K32: 32 input channels per matrix instruction, for 64 input channels.  (With
    // 32 the 16-channel form was the faster one, by 9%, in the kernel that gathered
    // its operands; in this one the other takes 394 us against 450, 32 -> 64 at
    // 128^3, but needs inputs of 16-byte alignment.)
    constexpr bool K32 = KT == 4;
    constexpr int CO = NT * 16, CI = KT * 16, RS = CI + (K32 ? 8 : 4);   // LDS row stride in BF16
    constexpr int CPS = CI / 8;                                          // 16-byte pieces of a site
    constexpr int NA = (kFwdSlots * CPS + kWsThreads - 1) / kWsThreads;  // pieces a thread stages per step: rows,
    constexpr int NW = (3 * CO * CPS + kWsThreads - 1) / kWsThreads;     // weights
    constexpr int OS = CO + 8;                                           // row stride of the output tile
    constexpr int IN = (kFwdSlots + 3 * CO) * RS, OUT = kFwdSites * OS;
    __shared__ __align__(16) uint16_t sBuf[IN > OUT ? IN : OUT];
    __shared__ int sSite[kFwdSites];           // site of each output row of the tile, from its first row on; -1: none
    __shared__ long long sRow[9][kFwdRows];    // first input element of each row's neighbour row at (dy, dz)
    uint16_t* const sX = sBuf;
    uint16_t* const sW = sBuf + kFwdSlots * RS;

    const ConvTile T = a.tile;
    // each XCD gets a contiguous run of tiles, whose neighbour rows share its L2
    const int qb = a.nblocks >> 3, rb = a.nblocks & 7, xcd = blockIdx.x & 7;
    const int blk = xcd * qb + min(xcd, rb) + (blockIdx.x >> 3);
    const int x0 = (blk % T.nseg) * T.w;
    const int ord = blk / T.nseg, in = (ord / (T.block * T.turns)) * T.block + ord % T.block;
    const int group = in + ord / T.block % T.turns * T.stride;
    if (in >= T.stride || group >= T.groups) return;   // a partial block or turn
    const long long r0 = (long long)group * T.rows, nrows = (long long)a.ly * a.lz;
    const int pitch = T.w + 2 * T.halo;   // staged sites of a row
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kq = lane >> 4, l16 = lane & 15;

    {
        const int r = tid / T.w, x = x0 + tid % T.w;
        sSite[tid] = (r < T.rows && r0 + r < nrows && x < a.lx) ? r * a.lx + x : -1;
    }
    for (int e = tid; e < 9 * kFwdRows; e += kWsThreads) {
        const int st = e / kFwdRows, r = e % kFwdRows;
        const long long row = r0 + r < nrows ? r0 + r : 0;
        const int y = wrapd(int(row % a.ly) + (st % 3 - 1) * a.dil, a.ly);
        const int z = wrapd(int(row / a.ly) + (st / 3 - 1) * a.dil, a.lz);
        sRow[st][r] = (y + (long long)a.ly * z) * a.lx * CI;
    }
    // slots of this lane's sites at dx = -1, 0, 1
    int off[kFwdMT][3];
#pragma unroll
    for (int mt = 0; mt < kFwdMT; ++mt) {
        const int m = wave * (16 * kFwdMT) + 16 * mt + l16;
        const int r = m / T.w, x = m % T.w;
        const bool in = r < T.rows;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int slot = x + T.halo;
            if (T.fold) slot = T.halo ? x + d * a.dil : wrapd(x + (d - 1) * a.dil, a.lx);
            off[mt][d] = in ? (r * pitch + slot) * RS : 0;
        }
    }
    // pieces this thread stages: LDS offset, row and first input element
    const int pieces = T.rows * pitch * CPS;
    int stOff[NA], stRow[NA], stX[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int e = tid + kWsThreads * i;
        const int slot = e / CPS, c = e % CPS, r = slot / pitch, p = slot % pitch;
        stOff[i] = e < pieces ? slot * RS + c * 8 : -1;
        stRow[i] = e < pieces ? r : 0;
        stX[i] = wrapd(x0 - T.halo + p, a.lx) * CI + c * 8;
    }
    const int steps = T.fold ? 9 : kTaps, tps = T.fold ? 3 : 1;
    const int wpieces = tps * CO * CPS;

    v4u ra[NA], rw[NW];
    auto get = [&](const uint16_t* src, bool vec) {
        if (vec) return *reinterpret_cast<const v4u*>(src);
        const uint2 lo = reinterpret_cast<const uint2*>(src)[0], hi = reinterpret_cast<const uint2*>(src)[1];
        return v4u{lo.x, lo.y, hi.x, hi.y};
    };
    auto load = [&](int step) {
        const long long* base = sRow[T.fold ? step : step / 3];
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (stOff[i] >= 0) {
                int x = stX[i];
                if (!T.fold) x = wrapd(x / CI + (step % 3 - 1) * a.dil, a.lx) * CI + x % CI;
                ra[i] = get(a.x + base[stRow[i]] + x, K32 || a.vecX);
            }
        const uint16_t* src = a.wt + (long long)step * tps * CO * CI;
#pragma unroll
        for (int i = 0; i < NW; ++i)
            if (tid + kWsThreads * i < wpieces) rw[i] = get(src + 8 * (tid + kWsThreads * i), a.vecW);
    };
    auto put = [&](uint16_t* dst, v4u v) {
        if constexpr (K32) {
            *reinterpret_cast<v4u*>(dst) = v;
        } else {   // rows of 8-byte alignment
            reinterpret_cast<uint2*>(dst)[0] = uint2{v[0], v[1]};
            reinterpret_cast<uint2*>(dst)[1] = uint2{v[2], v[3]};
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (stOff[i] >= 0) {
                v4u v = ra[i];
                if (a.reluIn) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = relu2(v[j]);
                }
                put(sX + stOff[i], v);
            }
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int e = tid + kWsThreads * i;
            if (e < wpieces) put(sW + (e / CPS) * RS + (e % CPS) * 8, rw[i]);
        }
    };

    v4f acc[kFwdMT][NT];
#pragma unroll
    for (int mt = 0; mt < kFwdMT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[mt][t] = v4f{0.f, 0.f, 0.f, 0.f};

    auto tap = [&](int d, const uint16_t* w) {
        if constexpr (K32) {
#pragma unroll
            for (int k2 = 0; k2 < KT / 2; ++k2) {
                v8bf av[kFwdMT];
#pragma unroll
                for (int mt = 0; mt < kFwdMT; ++mt)
                    av[mt] = __builtin_bit_cast(
                        v8bf, *reinterpret_cast<const v4u*>(sX + off[mt][d] + k2 * 32 + kq * 8));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const v8bf bv = __builtin_bit_cast(
                        v8bf, *reinterpret_cast<const v4u*>(w + (t * 16 + l16) * RS + k2 * 32 + kq * 8));
#pragma unroll
                    for (int mt = 0; mt < kFwdMT; ++mt)
                        acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[mt], bv, acc[mt][t], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                v4s av[kFwdMT];
#pragma unroll
                for (int mt = 0; mt < kFwdMT; ++mt)
                    av[mt] = __builtin_bit_cast(
                        v4s, *reinterpret_cast<const uint2*>(sX + off[mt][d] + kt * 16 + kq * 4));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const v4s bv = __builtin_bit_cast(
                        v4s, *reinterpret_cast<const uint2*>(w + (t * 16 + l16) * RS + kt * 16 + kq * 4));
#pragma unroll
                    for (int mt = 0; mt < kFwdMT; ++mt)
                        acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[mt], bv, acc[mt][t], 0, 0, 0);
                }
            }
        }
    };

    const long long site0 = r0 * a.lx;
    __syncthreads();   // sRow
    load(0);
    store();
    __syncthreads();
    for (int step = 0; step < steps; ++step) {
        if (step + 1 < steps) load(step + 1);
        tap(0, sW);
        if (T.fold) {
            tap(1, sW + CO * RS);
            tap(2, sW + 2 * CO * RS);
        }
        __syncthreads();
        if (step + 1 < steps) store();
        __syncthreads();
    }

    if (a.yf || !a.vecOut) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int co = t * 16 + l16;
            const float b = a.bias ? a.bias[co] : 0.f;
#pragma unroll
            for (int mt = 0; mt < kFwdMT; ++mt) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int site = sSite[wave * (16 * kFwdMT) + 16 * mt + 4 * kq + j];
                    if (site < 0) continue;
                    float v = acc[mt][t][j] + b;
                    const long long o = (site0 + site) * CO + co;
                    if (a.mask && !(bf2f(a.mask[o]) > 0.f)) v = 0.f;
                    if (a.yf)
                        a.yf[o] = v;
                    else
                        a.ybf[o] = f2bf(v);
                }
            }
        }
        return;
    }
    // BF16 output through LDS, so that it is stored (and the mask read) in
    // 16-byte pieces
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = t * 16 + l16;
        const float b = a.bias ? a.bias[co] : 0.f;
#pragma unroll
        for (int mt = 0; mt < kFwdMT; ++mt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                sBuf[(wave * (16 * kFwdMT) + 16 * mt + 4 * kq + j) * OS + co] = f2bf(acc[mt][t][j] + b);
    }
    __syncthreads();
    for (int e = tid; e < kFwdSites * (CO / 8); e += kWsThreads) {
        const int m = e / (CO / 8), c = e % (CO / 8), site = sSite[m];
        if (site < 0) continue;
        v4u v = *reinterpret_cast<const v4u*>(sBuf + m * OS + c * 8);
        const long long o = (site0 + site) * CO + c * 8;
        if (a.mask) {
            const v4u mk = *reinterpret_cast<const v4u*>(a.mask + o);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!(__uint_as_float(mk[j] << 16) > 0.f)) v[j] &= 0xffff0000u;
                if (!(__uint_as_float(mk[j] & 0xffff0000u) > 0.f)) v[j] &= 0xffffu;
            }
        }
        *reinterpret_cast<v4u*>(a.ybf + o) = v;
    }
}

// Tile of the forward kernel for a row length and dilation: the split of a row
// into equal segments that leaves the fewest of the work-group's site slots
// empty, staged sites included (whole rows need no halo: their neighbours wrap
// onto the row itself).  Where a halo of dil sites on both sides never fits,
// each tap's sites are staged by themselves.
inline ConvTile choose_conv_tile(int lx, int dil) {
    ConvTile best{};
    double bestCost = 1e300;
    for (int fold = 1; fold >= 0 && bestCost > 1e299; --fold)
        for (int nseg = 1; nseg <= lx; ++nseg) {
            const int w = (lx + nseg - 1) / nseg;
            if (w > kFwdSites) continue;
            if (w < 16 && nseg > 1) break;
            ConvTile t{w, (lx + w - 1) / w, 0, (fold && w < lx) ? dil : 0, fold};
            const long long pitch = w + 2LL * t.halo;
            if (pitch > kFwdSlots) continue;
            t.rows = int(std::min<long long>(std::min(kFwdSites / w, kFwdRows), kFwdSlots / pitch));
            // work-groups per row, and what their staging adds (9 reads per 27 taps of work)
            const double cost = double(t.nseg) / t.rows * (1.0 + 0.3 * double(t.rows * pitch) / kFwdSites);
            if (cost < bestCost) {
                bestCost = cost;
                best = t;
            }
        }
    return best;
}

// Order of the tiles, and the work-groups to launch for it.  64 -> 64 channels
// at 128^3 and dilation 4, where an XCD's L2 holds two planes: 0.67 ms against
// 0.77 in plain order; blocks of 8 or 32 row groups 0.68 and 0.69 ms.  The blocks
// are equal parts of a stride: whole ones of 16 left 15 of 16 work-groups without
// work where a plane is one row group (32 -> 64 channels, 16 x 16 x 4000, dilation
// 1: 824 us against 211).
inline int order_conv_tiles(ConvTile& t, int ly, int lz, int dil) {
    const long long rows = (long long)ly * lz;
    t.groups = int((rows + t.rows - 1) / t.rows);
    const long long apart = (long long)ly * std::min(dil, lz) / t.rows;
    t.stride = int(std::max<long long>(1, std::min<long long>(apart, t.groups)));
    t.turns = (t.groups + t.stride - 1) / t.stride;
    const int blocks = (t.stride + kFwdBlock - 1) / kFwdBlock;
    t.block = (t.stride + blocks - 1) / blocks;
    return int((long long)blocks * t.block * t.turns * t.nseg);
}

struct WgradArgs {
    const uint16_t* g;  // [n][cout] bf16 output gradient
    const uint16_t* x;  // [n][cin] bf16 layer input (before the layer's input ReLU)
    float* part;        // [slots][27][cout][cin]
    int cin, cout, lx, ly, lz, dil, reluIn;
    int pieces;             // 8-site pieces of a row (the last may be shorter)
    long long total, per;   // pieces of the lattice, and of one slot
    int slots, vec;         // vec: part is 16-byte aligned
};

constexpr int kWgSplit = 4;                         // waves that share a slot's sites for one tap
constexpr int kWgThreads = 3 * kWgSplit * 64;       // three taps
constexpr int kWgSites = 4096;                      // sites one wave adds up in FP32 at most
constexpr int kWgSlots = 28;                        // slots (of 9 work-groups) that 256 CUs run at once

// C / 16 consecutive channels of one site (2, 4 or 8 bytes): a lane's share of
// a 16-channel-group row
template <int PC>
struct Raw {
    unsigned w[PC == 4 ? 2 : 1];
};

template <int PC>
__device__ __forceinline__ Raw<PC> raw_load(const uint16_t* p) {
    Raw<PC> r;
    if constexpr (PC == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        r.w[0] = v.x;
        r.w[1] = v.y;
    } else if constexpr (PC == 2) {
        r.w[0] = *reinterpret_cast<const unsigned*>(p);
    } else {
        r.w[0] = *p;
    }
    return r;
}

// Channel c of eight sites as an operand of v_mfma_f32_16x16x32_bf16
template <int PC>
__device__ __forceinline__ v8bf raw_operand(const Raw<PC> (&r)[8], int c) {
    v4u v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = __builtin_amdgcn_perm(r[2 * i + 1].w[c >> 1], r[2 * i].w[c >> 1],
                                     (c & 1) ? 0x07060302u : 0x05040100u);
    return __builtin_bit_cast(v8bf, v);
}

// Weight gradient dW[tap][co][ci] = sum_site G[site][co] X[site + tap][ci]: a
// product whose contraction runs over the sites, while a site's channels are
// what lies together in memory.  A lane reads C / 16 consecutive channels of
// eight consecutive sites of a row and transposes them in registers, one byte
// permute per operand word: matrix row m of product a then stands for channel
// C / 16 m + a, which only the final store has to know.  So no operand passes
// through LDS, and the waves run without barriers until their sums are added.
// A work-group takes one slot of sites and the three taps of one (dy, dz),
// whose waves read the same G and, shifted by dil sites, the same X from the
// L1; four waves share a slot's sites per tap, and their sums are added in a
// fixed order through LDS.
// 64 x 64 channels of 302k sites: 160 us (418 TFLOP/s); staged in LDS per tap and
// transposed there by two-byte stores it took 770 us.  Bound by the operand
// loads through the L1 (8 KB per wave and 32 sites: one access in 73% of the
// clocks) and the vector work beside the 16 matrix instructions they feed (51%;
// the matrix cores 19%).
template <int NT, int KT>
__global__ void __launch_bounds__(kWgThreads) conv_wgrad_kernel(WgradArgs a) {
    constexpr int CO = NT * 16, CI = KT * 16;
    __shared__ __align__(16) float red[3][NT * KT][64][4];
    // each XCD gets whole slots: the nine (dy, dz) of a slot read the same sites
    const int nb = gridDim.x, qb = nb >> 3, rb = nb & 7, xcd = blockIdx.x & 7;
    const int blk = xcd * qb + min(xcd, rb) + (blockIdx.x >> 3);
    const int slot = blk / 9, dyz = blk % 9;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d = wave % 3, quarter = wave / 3;
    const int kq = lane >> 4, l16 = lane & 15;
    // the taps' offsets, wrapped into [0, length)
    const int dx = wrapd((d - 1) * a.dil, a.lx), dy = wrapd((dyz % 3 - 1) * a.dil, a.ly),
              dz = wrapd((dyz / 3 - 1) * a.dil, a.lz);

    const long long q0 = slot * a.per, q1 = min(a.total, q0 + a.per);
    long long q = q0 + 4 * quarter + kq;
    // x piece, y and z of the lane's piece, advanced by 4 kWgSplit pieces a turn
    int px = int(q % a.pieces), y = int(q / a.pieces % a.ly), z = int(q / a.pieces / a.ly);
    constexpr int kStride = 4 * kWgSplit;
    const int sx = kStride % a.pieces, sy = kStride / a.pieces % a.ly, sz = kStride / a.pieces / a.ly;

    v4f acc[NT][KT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int k = 0; k < KT; ++k) acc[i][k] = v4f{0.f, 0.f, 0.f, 0.f};

    const long long turns = (q1 - q0 + kStride - 1) / kStride;
    for (long long it = 0; it < turns; ++it, q += kStride) {
        const bool have = q < q1;
        const int x = have ? 8 * px : 0, yy = have ? y : 0, zz = have ? z : 0;
        const int valid = have ? min(8, a.lx - x) : 0;   // sites of this piece
        const uint16_t* gp = a.g + ((long long)x + (long long)a.lx * (yy + (long long)a.ly * zz)) * CO + NT * l16;
        const int yn = yy + dy >= a.ly ? yy + dy - a.ly : yy + dy, zn = zz + dz >= a.lz ? zz + dz - a.lz : zz + dz;
        const int xn = x + dx >= a.lx ? x + dx - a.lx : x + dx;
        const uint16_t* xp = a.x + (long long)a.lx * (yn + (long long)a.ly * zn) * CI + KT * l16;
        Raw<NT> g[8];
        Raw<KT> xv[8];
        if (__all(valid == 8 && xn + 8 <= a.lx)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) g[j] = raw_load<NT>(gp + j * CO);
            xp += (long long)xn * CI;
#pragma unroll
            for (int j = 0; j < 8; ++j) xv[j] = raw_load<KT>(xp + j * CI);
        } else {
            // a piece that ends with its row or wraps around it: sites past the end count as zeros
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const bool in = j < valid;
                int xs = xn + (in ? j : 0);
                xs = xs >= a.lx ? xs - a.lx : xs;
                g[j] = raw_load<NT>(gp + (in ? j : 0) * CO);
                xv[j] = raw_load<KT>(xp + (long long)xs * CI);
#pragma unroll
                for (unsigned& w : g[j].w) w = in ? w : 0u;
#pragma unroll
                for (unsigned& w : xv[j].w) w = in ? w : 0u;
            }
        }
        if (a.reluIn) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (unsigned& w : xv[j].w) w = relu2(w);
        }
        v8bf xb[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) xb[k] = raw_operand<KT>(xv, k);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const v8bf ga = raw_operand<NT>(g, i);
#pragma unroll
            for (int k = 0; k < KT; ++k)
                acc[i][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, xb[k], acc[i][k], 0, 0, 0);
        }
        px += sx;
        const int cx = px >= a.pieces;
        px -= cx ? a.pieces : 0;
        y += sy + cx;
        const int cy = y >= a.ly;
        y -= cy ? a.ly : 0;
        z += sz + cy;
    }
    for (int h = 1; h < kWgSplit; ++h) {
        if (quarter == h) {
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int k = 0; k < KT; ++k) *reinterpret_cast<v4f*>(red[d][i * KT + k][lane]) = acc[i][k];
        }
        __syncthreads();
        if (quarter == 0) {
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int k = 0; k < KT; ++k) acc[i][k] += *reinterpret_cast<const v4f*>(red[d][i * KT + k][lane]);
        }
        __syncthreads();
    }
    if (quarter != 0) return;
    // lane l, element j of acc[i][k] = dW[co = NT (4 (l / 16) + j) + i][ci = KT (l % 16) + k]
    const int tap = dyz * 3 + d;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float* o = a.part + (((long long)slot * kTaps + tap) * CO + NT * (4 * kq + j) + i) * CI + KT * l16;
            if (KT == 4 && a.vec) {
                *reinterpret_cast<v4f*>(o) = v4f{acc[i][0][j], acc[i][1 % KT][j], acc[i][2 % KT][j], acc[i][3 % KT][j]};
            } else {
#pragma unroll
                for (int k = 0; k < KT; ++k) o[k] = acc[i][k][j];
            }
        }
}

// Fixed-order sum over chunks.  A thread's loads are taken sixteen at a time,
// ahead of the additions: one after the other, 74 chunks of 27 x 64 x 64
// values took 69 us.
__global__ void wgrad_reduce_kernel(const float* part, long long chunks, long long per, float* out) {
    constexpr int kAhead = 16;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < per; e += (long long)gridDim.x * blockDim.x) {
        float s = 0.f;
        long long c = 0;
        for (; c + kAhead <= chunks; c += kAhead) {
            float v[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; ++k) v[k] = part[(c + k) * per + e];
#pragma unroll
            for (int k = 0; k < kAhead; ++k) s += v[k];
        }
        for (; c < chunks; ++c) s += part[c * per + e];
        out[e] = s;
    }
}

// Bias gradient, first stage: work-group b sums its chunk of sites for every
// channel, each thread eight channels of every (2048 / cout)th site (VEC; two
// bytes at a time where g is not 16-byte aligned); wgrad_reduce_kernel then
// adds the work-groups' rows in a fixed order.  302k sites of 64 channels:
// 8 us, two bytes at a time 44 us.
template <bool VEC>
__global__ void __launch_bounds__(kWsThreads) bias_grad_kernel(const uint16_t* g, long long n, int cout,
                                                              long long chunk, float* part) {
    constexpr int W = VEC ? 8 : 1;
    __shared__ float red[kWsThreads * W];
    const int cols = cout / W, rows = kWsThreads / cols, c = threadIdx.x % cols, r = threadIdx.x / cols;
    const long long s0 = (long long)blockIdx.x * chunk, s1 = min(n, s0 + chunk);
    float s[W];
#pragma unroll
    for (int k = 0; k < W; ++k) s[k] = 0.f;
#pragma unroll 4
    for (long long i = s0 + r; i < s1; i += rows) {
        if constexpr (VEC) {
            const v4u v = *reinterpret_cast<const v4u*>(g + i * cout + 8 * c);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                s[2 * k] += __uint_as_float(v[k] << 16);
                s[2 * k + 1] += __uint_as_float(v[k] & 0xffff0000u);
            }
        } else {
            s[0] += bf2f(g[i * cout + c]);
        }
    }
#pragma unroll
    for (int k = 0; k < W; ++k) red[(r * cols + c) * W + k] = s[k];
    __syncthreads();
    for (int e = threadIdx.x; e < cout; e += kWsThreads) {
        float t = 0.f;
        for (int k = 0; k < rows; ++k) t += red[k * cout + e];
        part[(long long)blockIdx.x * cout + e] = t;
    }
}

// Adam on FP32 master weights; refreshes the BF16 copy and, for [27][cout][cin]
// weights (cin > 0), the mirrored transpose used by the input gradient.
__global__ void adam_kernel(float* w, const float* g, float* m, float* v, long long count, float lr, float b1, float b2,
                            float eps, float c1, float c2, uint16_t* wbf, uint16_t* wbd, int cout, int cin) {
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += (long long)gridDim.x * blockDim.x) {
        const float gi = g[e];
        const float mi = b1 * m[e] + (1.f - b1) * gi;
        const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
        m[e] = mi;
        v[e] = vi;
        const float wi = w[e] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
        w[e] = wi;
        if (wbf) wbf[e] = f2bf(wi);
        if (wbd) {
            const long long per = (long long)cout * cin;
            const int tap = int(e / per), co = int((e / cin) % cout), ci = int(e % cin);
            wbd[((long long)(kTaps - 1 - tap) * cin + ci) * cout + co] = f2bf(wi);
        }
    }
}

// BF16 copies of FP32 weights (after initialisation or loading)
__global__ void weights_to_bf16_kernel(const float* w, long long count, uint16_t* wbf, uint16_t* wbd, int cout, int cin) {
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += (long long)gridDim.x * blockDim.x) {
        const uint16_t b = f2bf(w[e]);
        wbf[e] = b;
        if (wbd) {
            const long long per = (long long)cout * cin;
            const int tap = int(e / per), co = int((e / cin) % cout), ci = int(e % cin);
            wbd[((long long)(kTaps - 1 - tap) * cin + ci) * cout + co] = b;
        }
    }
}

// Offset added to the first five output channels: the network predicts Q as a
// correction to the uniform far-field state.
struct Off5 {
    float v[5];
};

// Gradient of the mean squared error over liquid-crystal sites (types <= 0) on
// the first five output channels (plus the offset); per-block partial losses in FP64.
__global__ void __launch_bounds__(kWsThreads) mse_grad_kernel(const float* y, int cy, const float* target,
                                                             const int8_t* types, long long n, float scale,
                                                             uint16_t* g, double* lossPart, Off5 off) {
    __shared__ double red[kWsThreads];
    double l = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const bool lc = types[i] <= 0;
        for (int c = 0; c < cy; ++c) {
            float gv = 0.f;
            if (lc && c < 5) {
                const float d = (y[i * cy + c] + off.v[c]) - target[i * 5 + c];
                l += double(d) * double(d);
                gv = 2.f * d * scale;
            }
            g[i * cy + c] = f2bf(gv);
        }
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int w = kWsThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) lossPart[blockIdx.x] = red[0];
}

// Energy term of the training loss: g[s][c] -= scale F_c(s) for the first five
// channels of liquid-crystal sites, F being the force computer's force on the
// predicted state (minus the energy gradient, shaped by the metric).
template <typename R>
__global__ void __launch_bounds__(kWsThreads) energy_grad_kernel(const R* f, const SiteType* types, long long n,
                                                               int cy, float scale, uint16_t* g) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        if (types[i] > 0) continue;
#pragma unroll
        for (int c = 0; c < 5; ++c) g[i * cy + c] = f2bf(bf2f(g[i * cy + c]) - scale * float(f[c * n + i]));
    }
}

// Input features, channels-last [n][16] bf16:
//  0-2 one-hot of bulk / next to an object / object,
//  3-7 anchoring tensor of object sites: Q^B / S0 for homeotropic objects,
//      -(nu nu - I/3) for degenerate planar (nu = the first three entries of Q^B),
//  8   planar flag, 9 log(W) / 3 (object sites),
//  10-14 far-field tensor d d - I/3 (every site), 15 zero.
template <typename R>
__global__ void features_kernel(const R* q, const SiteType* types, const DevObject* objects, long long n, double dx,
                                double dy, double dz, uint16_t* out) {
    const float far[5] = {float(dx * dx - 1.0 / 3.0), float(dx * dy), float(dx * dz), float(dy * dy - 1.0 / 3.0),
                          float(dy * dz)};
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        float f[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) f[c] = 0.f;
        const int t = types[i];
        f[t == 0 ? 0 : (t < 0 ? 1 : 2)] = 1.f;
        if (t > 0) {
            const DevObject o = objects[t - 1];
            float qb[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) qb[c] = float(q[c * n + i]);
            if (o.type == 0) {
                const float s = o.P2 != 0 ? float(1.0 / o.P2) : 1.f;
#pragma unroll
                for (int c = 0; c < 5; ++c) f[3 + c] = qb[c] * s;
            } else {
                const float nx = qb[0], ny = qb[1], nz = qb[2];
                f[3] = -(nx * nx - 1.f / 3.f);
                f[4] = -nx * ny;
                f[5] = -nx * nz;
                f[6] = -(ny * ny - 1.f / 3.f);
                f[7] = -ny * nz;
                f[8] = 1.f;
            }
            f[9] = o.P1 > 0 ? float(log(o.P1) / 3.0) : 0.f;
        }
#pragma unroll
        for (int c = 0; c < 5; ++c) f[10 + c] = far[c];
#pragma unroll
        for (int c = 0; c < 16; ++c) out[i * 16 + c] = f2bf(f[c]);
    }
}

// Q of liquid-crystal sites from the first five channels of y; velocities zero.
__global__ void types_to_i8_kernel(const SiteType* types, long long n, int8_t* out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        out[i] = int8_t(types[i] > 127 ? 127 : types[i]);
}

template <typename R>
__global__ void apply_kernel(const float* y, int cy, const SiteType* types, long long n, R* q, R* u, Off5 off) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        if (types[i] <= 0) {
#pragma unroll
            for (int c = 0; c < 5; ++c) q[c * n + i] = R(y[i * cy + c] + off.v[c]);
        }
#pragma unroll
        for (int c = 0; c < 5; ++c) u[c * n + i] = R(0);
    }
}

template <typename R>
__global__ void extract_q_kernel(const R* q, long long n, float* out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 5; ++c) out[i * 5 + c] = float(q[c * n + i]);
    }
}

inline int grid_for(long long work, int per = kWsThreads) {
    long long b = (work + per - 1) / per;
    return int(b < 1 ? 1 : (b > 65536 ? 65536 : b));
}

template <int NT, int KT>
hipError_t launch_fwd_t(const ConvArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((conv_fwd_kernel<NT, KT>), dim3(a.nblocks), dim3(kWsThreads), 0, s, a);
    return hipGetLastError();
}

template <int NT, int KT>
hipError_t launch_wgrad_t(const WgradArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((conv_wgrad_kernel<NT, KT>), dim3(9 * a.slots), dim3(kWgThreads), 0, s, a);
    return hipGetLastError();
}

// channel counts supported: multiples of 16 up to 64
#define QMIN_WS_DISPATCH(FN, NT_, KT_, ...)                                        \
    switch ((NT_) * 8 + (KT_)) {                                                  \
        case 1 * 8 + 1: return FN<1, 1>(__VA_ARGS__);                             \
        case 1 * 8 + 2: return FN<1, 2>(__VA_ARGS__);                             \
        case 1 * 8 + 4: return FN<1, 4>(__VA_ARGS__);                             \
        case 2 * 8 + 1: return FN<2, 1>(__VA_ARGS__);                             \
        case 2 * 8 + 2: return FN<2, 2>(__VA_ARGS__);                             \
        case 2 * 8 + 4: return FN<2, 4>(__VA_ARGS__);                             \
        case 4 * 8 + 1: return FN<4, 1>(__VA_ARGS__);                             \
        case 4 * 8 + 2: return FN<4, 2>(__VA_ARGS__);                             \
        case 4 * 8 + 4: return FN<4, 4>(__VA_ARGS__);                             \
        default: return hipErrorInvalidValue;                                     \
    }

hipError_t launch_fwd(const ConvArgs& a, hipStream_t s) { QMIN_WS_DISPATCH(launch_fwd_t, a.cout / 16, a.cin / 16, a, s) }

hipError_t launch_wgrad(const WgradArgs& a, hipStream_t s) {
    QMIN_WS_DISPATCH(launch_wgrad_t, a.cout / 16, a.cin / 16, a, s)
}

bool channels_ok(int c) { return c == 16 || c == 32 || c == 64; }

}  // namespace ws
}  // namespace qmin

using namespace qmin;
using namespace qmin::ws;

extern "C" {

int qm_ws_conv_forward(const void* x, int cin, const void* wt, const float* bias, int cout, const void* mask,
                       void* ybf16, float* yf32, int lx, int ly, int lz, int dil, int reluIn, void* stream) {
    if (!channels_ok(cin) || !channels_ok(cout)) return fail(QM_EINVAL, "channels must be 16, 32 or 64");
    if (!x || !wt || (!ybf16 && !yf32) || lx < 1 || ly < 1 || lz < 1 || dil < 1)
        return fail(QM_EINVAL, "bad convolution argument");
    ConvArgs a{};
    a.x = static_cast<const uint16_t*>(x);
    a.wt = static_cast<const uint16_t*>(wt);
    a.bias = bias;
    a.mask = static_cast<const uint16_t*>(mask);
    a.ybf = static_cast<uint16_t*>(ybf16);
    a.yf = yf32;
    a.n = (long long)lx * ly * lz;
    a.cin = cin;
    a.cout = cout;
    a.lx = lx;
    a.ly = ly;
    a.lz = lz;
    a.dil = dil;
    a.reluIn = reluIn;
    a.tile = choose_conv_tile(lx, dil);
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    a.vecX = aligned(x);
    a.vecW = aligned(wt);
    a.vecOut = aligned(ybf16) && aligned(mask);
    a.nblocks = order_conv_tiles(a.tile, ly, lz, dil);
    HIP_TRY(launch_fwd(a, static_cast<hipStream_t>(stream)));
    return QM_OK;
}

int qm_ws_conv_wgrad(const void* g, int cout, const void* x, int cin, int reluIn, int lx, int ly, int lz, int dil,
                     float* part, long long chunk, float* dw, void* stream) {
    if (!channels_ok(cin) || !channels_ok(cout)) return fail(QM_EINVAL, "channels must be 16, 32 or 64");
    if (!g || !x || !part || !dw || lx < 1 || ly < 1 || lz < 1 || chunk < 16 || chunk % 16)
        return fail(QM_EINVAL, "bad weight-gradient argument");
    WgradArgs a{};
    a.g = static_cast<const uint16_t*>(g);
    a.x = static_cast<const uint16_t*>(x);
    a.part = part;
    a.cin = cin;
    a.cout = cout;
    a.lx = lx;
    a.ly = ly;
    a.lz = lz;
    a.dil = dil;
    a.reluIn = reluIn;
    a.vec = (reinterpret_cast<uintptr_t>(part) & 15) == 0;
    a.pieces = (lx + 7) / 8;
    a.total = (long long)a.pieces * ly * lz;
    // part holds one row of partial sums per chunk: as many slots of sites at
    // most; fewer where a whole number of rounds over the CUs already keeps
    // every wave's FP32 sum within kWgSites sites
    const long long n = (long long)lx * ly * lz, chunks = (n + chunk - 1) / chunk;
    const long long rounds = (n + (long long)kWgSites * kWgSplit * kWgSlots - 1) / ((long long)kWgSites * kWgSplit * kWgSlots);
    a.slots = int(std::min(chunks, kWgSlots * rounds));
    a.per = (a.total + a.slots - 1) / a.slots;
    hipStream_t s = static_cast<hipStream_t>(stream);
    HIP_TRY(launch_wgrad(a, s));
    const long long per = (long long)kTaps * cout * cin;
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(grid_for(per)), dim3(kWsThreads), 0, s, part, (long long)a.slots, per, dw);
    HIP_TRY(hipGetLastError());
    return QM_OK;
}

int qm_ws_bias_grad(const void* g, long long n, int cout, float* part, int blocks, float* db, void* stream) {
    if (!g || !db || !part || !channels_ok(cout) || blocks < 1 || n < 1) return fail(QM_EINVAL, "bad argument");
    const long long chunk = (n + blocks - 1) / blocks;
    const auto st = static_cast<hipStream_t>(stream);
    const bool vec = (reinterpret_cast<uintptr_t>(g) & 15) == 0;
    hipLaunchKernelGGL(vec ? bias_grad_kernel<true> : bias_grad_kernel<false>, dim3(blocks), dim3(kWsThreads), 0, st,
                       static_cast<const uint16_t*>(g), n, cout, chunk, part);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(1), dim3(64), 0, st, part, (long long)blocks, (long long)cout, db);
    HIP_TRY(hipGetLastError());
    return QM_OK;
}

int qm_ws_adam(float* w, const float* g, float* m, float* v, long long count, float lr, float b1, float b2, float eps,
               int step, void* wbf16, void* wbd16, int cout, int cin, void* stream) {
    if (!w || !g || !m || !v || step < 1) return fail(QM_EINVAL, "bad argument");
    const float c1 = 1.f / (1.f - powf(b1, float(step))), c2 = 1.f / (1.f - powf(b2, float(step)));
    hipLaunchKernelGGL(adam_kernel, dim3(grid_for(count)), dim3(kWsThreads), 0, static_cast<hipStream_t>(stream), w, g,
                       m, v, count, lr, b1, b2, eps, c1, c2, static_cast<uint16_t*>(wbf16),
                       static_cast<uint16_t*>(wbd16), cout, cin);
    HIP_TRY(hipGetLastError());
    return QM_OK;
}

int qm_ws_weights_to_bf16(const float* w, long long count, void* wbf16, void* wbd16, int cout, int cin, void* stream) {
    if (!w || !wbf16) return fail(QM_EINVAL, "bad argument");
    hipLaunchKernelGGL(weights_to_bf16_kernel, dim3(grid_for(count)), dim3(kWsThreads), 0,
                       static_cast<hipStream_t>(stream), w, count, static_cast<uint16_t*>(wbf16),
                       static_cast<uint16_t*>(wbd16), cout, cin);
    HIP_TRY(hipGetLastError());
    return QM_OK;
}

static Off5 off5(const double* offset5) {
    Off5 o{};
    for (int c = 0; c < 5; ++c) o.v[c] = offset5 ? float(offset5[c]) : 0.f;
    return o;
}

int qm_ws_mse_grad(const float* y, int cy, const float* target, const void* types, long long n, float scale,
                   const double* offset5, void* g, double* lossPart, int blocks, void* stream) {
    if (!y || !target || !types || !g || !lossPart || blocks < 1 || cy < 5) return fail(QM_EINVAL, "bad argument");
    hipLaunchKernelGGL(mse_grad_kernel, dim3(blocks), dim3(kWsThreads), 0, static_cast<hipStream_t>(stream), y, cy,
                       target, static_cast<const int8_t*>(types), n, scale, static_cast<uint16_t*>(g), lossPart,
                       off5(offset5));
    HIP_TRY(hipGetLastError());
    return QM_OK;
}

// The energy term of the warm-start loss: the lattice holds the prediction
// (qm_ws_apply); its forces are computed and -scale F added to the first five
// channels of g at liquid-crystal sites.  The caller's stream is drained first.
int qm_ws_energy_grad(qm_ldg* f, qm_lattice* L, float scale, void* g, int cy, void* stream) {
    if (!f || !L || !g || cy < 5) return fail(QM_EINVAL, "bad argument");
    HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    if (int rc = qm_ldg_compute_forces(f, L)) return rc;
    const int blocks = grid_for(L->n);
    if (L->precision == QM_FP64)
        hipLaunchKernelGGL(energy_grad_kernel<double>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<double>(L, L->hCtrl.cur).f, L->dTypes, L->n, cy, scale,
                           static_cast<uint16_t*>(g));
    else
        hipLaunchKernelGGL(energy_grad_kernel<float>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<float>(L, L->hCtrl.cur).f, L->dTypes, L->n, cy, scale,
                           static_cast<uint16_t*>(g));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(L->stream));
    return QM_OK;
}

// features of a lattice's current geometry; out is [n][16] bf16 on the device
int qm_ws_features(qm_lattice* L, double dx, double dy, double dz, void* out) {
    if (!L || !out) return fail(QM_EINVAL, "bad argument");
    if (int rc = sync_ctrl_to_host(L)) return rc;
    const int blocks = grid_for(L->n);
    if (L->precision == QM_FP64)
        hipLaunchKernelGGL(features_kernel<double>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<double>(L, L->hCtrl.cur).q, L->dTypes, L->dObjects, L->n, dx, dy, dz,
                           static_cast<uint16_t*>(out));
    else
        hipLaunchKernelGGL(features_kernel<float>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<float>(L, L->hCtrl.cur).q, L->dTypes, L->dObjects, L->n, dx, dy, dz,
                           static_cast<uint16_t*>(out));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(L->stream));
    return QM_OK;
}

// the device site types as int8 (reference encoding, object ids above 127 clamped
// to 127: the network's inputs and loss only tell objects from the rest)
int qm_ws_types(qm_lattice* L, void* out) {
    if (!L || !out) return fail(QM_EINVAL, "bad argument");
    hipLaunchKernelGGL(types_to_i8_kernel, dim3(grid_for(L->n)), dim3(kWsThreads), 0, L->stream, L->dTypes, L->n,
                       static_cast<int8_t*>(out));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(L->stream));
    return QM_OK;
}

// Q of liquid-crystal sites from y (first five of cy channels, FP32, device)
// plus offset5 (host, may be NULL); velocities are cleared and any pending FIRE
// velocity mix dropped
int qm_ws_apply(qm_lattice* L, const float* y, int cy, const double* offset5) {
    if (!L || !y || cy < 5) return fail(QM_EINVAL, "bad argument");
    if (int rc = sync_ctrl_to_host(L)) return rc;
    const int blocks = grid_for(L->n);
    if (L->precision == QM_FP64) {
        const StateSet<double> st = state_set<double>(L, L->hCtrl.cur);
        hipLaunchKernelGGL(apply_kernel<double>, dim3(blocks), dim3(kWsThreads), 0, L->stream, y, cy, L->dTypes, L->n,
                           st.q, st.u, off5(offset5));
    } else {
        const StateSet<float> st = state_set<float>(L, L->hCtrl.cur);
        hipLaunchKernelGGL(apply_kernel<float>, dim3(blocks), dim3(kWsThreads), 0, L->stream, y, cy, L->dTypes, L->n,
                           st.q, st.u, off5(offset5));
    }
    HIP_TRY(hipGetLastError());
    L->hCtrl.identity = 1;
    L->hCtrl.reset = 0;
    if (int rc = push_ctrl(L)) return rc;
    HIP_TRY(hipStreamSynchronize(L->stream));
    return QM_OK;
}

// current Q as FP32 [n][5] on the device
int qm_ws_extract_q(qm_lattice* L, float* out) {
    if (!L || !out) return fail(QM_EINVAL, "bad argument");
    if (int rc = sync_ctrl_to_host(L)) return rc;
    const int blocks = grid_for(L->n);
    if (L->precision == QM_FP64)
        hipLaunchKernelGGL(extract_q_kernel<double>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<double>(L, L->hCtrl.cur).q, L->n, out);
    else
        hipLaunchKernelGGL(extract_q_kernel<float>, dim3(blocks), dim3(kWsThreads), 0, L->stream,
                           state_set<float>(L, L->hCtrl.cur).q, L->n, out);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(L->stream));
    return QM_OK;
}

}  // extern "C"
