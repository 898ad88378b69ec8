// Lattice passes of the Adam and Nesterov iterations: the fused and boundary
// passes in modes kAdamStep / kNesterovStep compute each site's force and then
// apply the minimizer's update to that site (energyMinimizerAdam.cpp:25-54,
// energyMinimizerNesterovAG.cpp:75-92), writing the new Q and the force to the
// other state set and the work-group partial sums of |F|^2 to the lattice's
// partials.  One pass per iteration: the update needs only the site's own
// force and its own entries of the minimizer's vectors, so it rides on the
// store of the force instead of a second pass over Q, F and those vectors.
#include "lattice_pass.h"

namespace qmin {
// Queues the fused pass (tile `tile`, one of the halo-padded ones or kBlock) and
// the boundary pass of one Adam or Nesterov iteration.
template <typename R>
hipError_t launch_step(const MarchArgs<R>& ma, const BoundaryArgs<R>& ba, int mode, int terms, int tile,
                       hipStream_t s) {
    if (!(tile >= 0 && tile < kNumMarchTiles) && tile != kBlock) return hipErrorInvalidValue;
    if (!is_step_mode(mode)) return hipErrorInvalidValue;
    const void* fn = mode == kAdamStep ? march_fn_mode<R, kAdamStep>(terms, tile, ma.nt != 0)
                                       : march_fn_mode<R, kNesterovStep>(terms, tile, ma.nt != 0);
    void* margs[] = {const_cast<MarchArgs<R>*>(&ma)};
    hipError_t e = hipLaunchKernel(fn, dim3(ma.nblocks), dim3(tile_threads(tile)), margs, 0, s);
    if (e != hipSuccess) return e;
    const bool lanes = boundary_lanes(terms, ba.nsites);
    const int blocks = boundary_blocks(ba.nsites, lanes);
    if (blocks == 0) return hipGetLastError();
    const void* bfn = mode == kAdamStep ? boundary_fn<R, kAdamStep>(terms, lanes) : boundary_fn<R, kNesterovStep>(terms, lanes);
    void* bargs[] = {const_cast<BoundaryArgs<R>*>(&ba)};
    e = hipLaunchKernel(bfn, dim3((unsigned)blocks), dim3(kBoundaryThreads), bargs, 0, s);
    if (e != hipSuccess) return e;
    return hipGetLastError();
}

template hipError_t launch_step<double>(const MarchArgs<double>&, const BoundaryArgs<double>&, int, int, int,
                                        hipStream_t);
template hipError_t launch_step<float>(const MarchArgs<float>&, const BoundaryArgs<float>&, int, int, int,
                                       hipStream_t);

}  // namespace qmin
