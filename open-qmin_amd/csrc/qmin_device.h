// Shared host/device definitions of the qmin HIP library (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qmin {

// Work-group of the fused pass: one thread per site of a TX x TY tile with a
// one-site halo in x and y; the work-group marches along z through a chunk.
// Four tile shapes are compiled: 32 x 8 and 64 x 4 (256 threads; wider rows use
// whole cache lines for the side halo but have more halo sites per tile), and
// 32 x 16 and 64 x 8 (512 threads, 73-79 KB of LDS in FP64: fewer halo sites per
// site; with 64 x 8 each wave covers one contiguous 64-site row).
// Tiles 4..6 are those of the FIRE pass that keeps only Q and v between
// iterations (fire_stream.hip): TX x TY owned sites, one thread per site of the
// tile plus a two-site margin.
constexpr int kThreads = 256;   // work-group size of the streaming kernels
enum TileId {
    kTile32x8 = 0, kTile64x4 = 1, kTile32x16 = 2, kTile64x8 = 3, kNumMarchTiles = 4,
    kStream32x16 = 4, kStream32x8 = 5, kStream64x8 = 6, kNumTiles = 7,
    kBlock = 7
};
constexpr int kTileTX[kNumTiles] = {32, 64, 32, 64, 32, 32, 64};
constexpr int kTileTY[kNumTiles] = {8, 4, 16, 8, 16, 8, 8};
constexpr int kTileThreads[kNumMarchTiles] = {32 * 8, 64 * 4, 32 * 16, 64 * 8};
__host__ __device__ constexpr bool is_stream_tile(int tile) { return tile >= kNumMarchTiles && tile < kNumTiles; }

// Block of the fused pass on small lattices (kBlock, automatic only): sites a
// work-group owns in x, y and z at most, one thread per site.
struct Block {
    static constexpr int BX = 16, BY = 4, BZ = 4;
    static constexpr int Threads = BX * BY * BZ;
    static constexpr int HX = BX + 2, HP = HX * (BY + 2), HZ = BZ + 2;   // halo-padded rows, planes and planes' count
    static constexpr int Halo = HP * HZ - Threads;
};

// Rows of a tile at most in an ensemble's pass.  Where a lattice's rows are
// shorter than TX, the threads this leaves over take more rows: a quarter more
// than TY in FP32 (40 lattices of 24 to 96 sites, 64 x 4 tiles: 246 against 287
// us per iteration).  In FP64 the planes of those rows would cost a work-group
// per CU in LDS, and TY is the most.
template <typename R>
constexpr int tile_rows(int tile) {
    return sizeof(R) == 4 ? kTileTY[tile] * 5 / 4 : kTileTY[tile];
}

// threads of a work-group of the fused pass
inline int tile_threads(int tile) { return tile == kBlock ? Block::Threads : kTileThreads[tile]; }

struct TileGrid {
    int tw, th;      // sites of a tile in x and y
    int nbx, nby;    // tiles in x and y
};

// Tiles of one lattice plane; narrow: rows shorter than TX make room for more of
// them, up to rowsMax.
inline TileGrid tile_grid(int lx, int ly, int tile, bool narrow = false, int rowsMax = 0) {
    auto parts = [](int l, int most) { return (l + most - 1) / most; };
    if (tile == kBlock) {
        TileGrid g{0, 0, parts(lx, Block::BX), parts(ly, Block::BY)};
        g.tw = parts(lx, g.nbx);
        g.th = parts(ly, g.nby);
        return g;
    }
    const int tx = kTileTX[tile], ty = kTileTY[tile];
    TileGrid g{tx, ty, parts(lx, tx), parts(ly, ty)};
    // (Longer rows are not cut into equal parts: 203 sites in tiles of 51 instead
    // of 64 took 316 against 285 us in FP32, with a fifth fewer tiles, as more
    // cache lines are shared between tiles and written in parts.)
    if (!narrow || g.nbx > 1) return g;
    g.tw = lx;
    g.th = tx * ty / g.tw < rowsMax ? tx * ty / g.tw : rowsMax;
    g.nby = parts(ly, g.th);
    g.th = parts(ly, g.nby);
    return g;
}

template <int TX_, int TY_, int Rows>
struct Tile {
    static constexpr int TX = TX_, TY = TY_;
    static constexpr int Threads = TX * TY;        // one site per thread
    static constexpr int HX = TX + 2;              // row pitch of one halo-padded plane
    static constexpr int HP = HX * (Rows + 2);     // sites of it
    static_assert(Threads % 64 == 0, "whole wave64s");
    static_assert(2 * HX + 2 * Rows <= Threads, "one halo site per thread at most");
};

using SiteType = int16_t;                // site types on the device (reference encoding)
constexpr int kMaxObjects = 32767;      // object ids a SiteType holds
constexpr int kBoundaryThreads = 128;
constexpr int kBoundaryLanes = 8;   // lanes that evaluate one site together, where the pass does so
constexpr int kBoundaryGroup = kBoundaryThreads / kBoundaryLanes;   // sites of such a work-group
constexpr int kBoundaryCases = 27;

// Whether the boundary pass gives a site eight lanes (boundary_lanes_body) or one
// (boundary_site_body).  Few sites leave the chip idle, and the length of one
// wave's path decides: lanes.  Many fill it, and the loads, which eight lanes
// scatter over more lines, set the pace.  FIRE iterations with lanes less those
// with one lane per site (us; walls across z, then spheres; FP64 / FP32):
//   L1      6,400 sites  -4 / -3 (spheres), 16,200  +1 / +0.5, 18,400  +2 / +1
//           and +1 / 0, 32,800  +4 / +3, 80,000  +11 / +9, 131,000  +19 / +15
//   L1..L3  6,400  -10 / -11 (spheres), 16,200  0 / -1, 18,400  +2 / 0 and
//           0 / 0, 33,000  +6 / +4, 80,000  +17 / +13 and (83,000) 0 / +9
//   L1..L6  6,400  -27 / -23 (spheres), 16,200  -1 / -1, 18,400  +2 / +2 and
//           -7 / -3, 22,800  +1 / +8 (spheres), 33,000  +8 / +7, 41,000  +14 / +26
//           (spheres), 131,000  +42 / +43
// Ensembles, by the sum of their lattices' sites: the same line, to 4%.
constexpr long long kLanesSitesOne = 16384, kLanesSites = 18432;
inline bool boundary_lanes(int terms, long long nsites) {
    return nsites <= (terms == 0 ? kLanesSitesOne : kLanesSites);
}
// work-groups of the boundary pass over nsites sites
inline int boundary_blocks(long long nsites, bool lanes) {
    const int per = lanes ? kBoundaryGroup : kBoundaryThreads;
    return int((nsites + per - 1) / per);
}

// One term of a boundary stencil, at unit constants: coefficient(s) and the
// inputs multiplied (the 125 of a site, then the constant 1).
struct BoundaryLinTerm {
    double c2, c3, c4;
    short a, b;
};
struct BoundaryQuadTerm {
    double c6;
    short a, b;
};

// The same composed for a force's constants in the lattice's precision, as the
// boundary pass reads it: [case][component][round][lane], the terms of L2..L4
// first, those of L6 behind them.
template <typename R>
struct BoundaryTerm {
    R coef;
    int ab;   // a + 256 b
};

constexpr int kReduceThreads = 256;
constexpr int kMaxEnergyBlocks = 4096;
constexpr int kFastWeights = 160;  // >= entries of the composed L1..L4 operator

// kAdamStep, kNesterovStep: the force of every site, then that minimizer's
// update of the site, written to the other state set (one pass per iteration)
enum Mode { kForce = 0, kFire = 1, kAdamStep = 2, kNesterovStep = 3 };
// kMultiLinear: L1..L3, kMultiL4: L1..L4, kMultiL6: L1..L4 and L6
enum Terms { kOneConstant = 0, kMultiLinear = 1, kMultiL4 = 2, kMultiL6 = 3 };

struct DevObject {
    int type;  // 0 homeotropic, 1 degenerate planar
    int pad;
    double P1, P2;
};

struct ForceConst {
    double a, b, c;        // A/2, B/3, C/4 of the phase energy
    double L1, L2, L3, L4, L6;
    double field[5];       // uniform E and H field force, added to the raw force
    int hasField;
    int semantics;         // 0 reference CPU two-pass, 1 reference GPU single pass
};

// Device-resident control block of one lattice: which state set is current and
// the FIRE scalars, advanced by the last work-group of each iteration.
struct Ctrl {
    int cur;
    int done;
    int iterations;
    int maxIter;
    int nPositive;
    int reset;      // pending velocity reset (v = 0) from the last FIRE step
    int identity;   // no pending velocity mix (v = u)
    int nanFlag;
    int traceLen;
    int traceCap;
    double dt, alpha;
    double cKeep, cForce;   // pending mix v = cKeep u + cForce F
    double forceMax, power, fnorm, vnorm, scaling;
};

struct FireConst {
    double alphaStart, dtMax, dtInc, dtDec, alphaDec, alphaMin, dtMin, fc, nTotal;
    int nMin;
    int pad;
};

struct EnergyConst {
    double a, b, c;
    double L[5];  // L1, L2, L3, L4, L6
    int eOn, hOn;
    double E[3], eps, eps0, deps;
    double H[3], chi, mu0, dchi;
    const double* hvar;   // spatially varying H, planes hx, hy, hz of n (null: none)
};

// The Adam or Nesterov update that a pass in mode kAdamStep / kNesterovStep
// applies to each site once its force is known.
struct StepArgs {
    void* m;             // Adam: first moment; Nesterov: the alternate sequence (5 planes of n, lattice precision)
    void* v;             // Adam: second moment
    const double* scal;  // device scalars: Adam beta1^t, beta2^t; Nesterov lambda, mu
    double dt, b1, b2, eps;
    int scheduled;       // Nesterov: momentum 1 + gamma from lambda
    int pad;
};

template <typename R>
struct StateSet {
    R* q;  // 5 planes of n
    R* u;
    R* f;
};

// A FIRE pass that begins with the scalar step of the iteration before it, whose
// partial sums are then still to be summed (block_body): an iteration is one
// launch less.  The control block alternates between two places, as some
// work-groups read the old one while the first writes the new.
struct ChainArgs {
    int on;                 // the pass is one of these
    int pending;            // there is such a step (not before a run's first pass)
    int cur;                // the current state set, unless the run is done
    const double* prev;     // partial sums of the previous iteration
    long long total;        // and their slots
    Ctrl* next;             // receives the control block after the step
    FireConst fire;
    double* trace;
};

template <typename R>
struct MarchArgs {
    StateSet<R> set[2];
    const int8_t* cls;      // per site: 0 composed bulk formula, > 0 object, < 0 finished by the boundary pass
    int gate;               // force-only pass: skip once the control block reports done
    int lx, ly, lz, zchunk;
    long long n;
    int nbx, nby, nblocks;
    int tw, th;             // sites of a tile in x and y (tile_grid)
    ForceConst fc;
    Ctrl* ctrl;
    double* partials;   // [nblocks + boundary blocks][3]
    const R* W;         // composed bulk operator weights (device buffer, read with scalar loads)
    const double* hvar; // spatially varying H, planes hx, hy, hz of n (null: none)
    double hvarP;       // deltaChi mu0
    int storeF;         // FIRE pass that keeps only Q and v, and the Adam and Nesterov passes: store F of the sites
                        // they finish as well
    int nt;             // non-temporal stores of the next state (marching passes)
    StepArgs step;      // modes kAdamStep, kNesterovStep
    ChainArgs chain;    // block pass in mode kFire
};

template <typename R>
struct BoundaryArgs {
    StateSet<R> set[2];
    const SiteType* types;
    const DevObject* objects;
    const int32_t* sites;   // compacted list of sites finished here
    int gate;
    long long nsites;
    int lx, ly, lz;
    long long n;
    const BoundaryTerm<R>* terms;   // stencils of the 27 cases for the force's constants
    int marchBlocks;        // partial slots used by the fused pass
    ForceConst fc;
    FireConst fire;
    Ctrl* ctrl;
    double* partials;
    double* trace;          // [traceCap][6]
    const double* hvar;
    double hvarP;
    StepArgs step;          // modes kAdamStep, kNesterovStep
};

// Per-lattice arguments of the batched FIRE scalar step.
struct FinalizeDesc {
    Ctrl* ctrl;
    FireConst fire;
    const double* partials;
    long long total;
};

struct EnsembleStatus {
    int done;
    int iterations;
    double forceMax;
};

}  // namespace qmin
