// The tiled MUSCL step (zfv_tile.hpp) with the HLL and Rusanov fluxes.
#include "zfv_tile.hpp"

namespace zfv {

hipError_t launch_tile_hll(int limiter, int variant, const TileMesh& T, const DevState& in, const DevState& out,
                           const int* wait_in, int* wait_out, const Eos& eos, const StepCtl& ctl, hipStream_t s) {
    return launch_tile_flux<2>(limiter, variant, false, T, in, out, wait_in, wait_out, eos, ctl, s);
}

hipError_t launch_tile_rusanov(int limiter, int variant, const TileMesh& T, const DevState& in, const DevState& out,
                               const int* wait_in, int* wait_out, const Eos& eos, const StepCtl& ctl, hipStream_t s) {
    return launch_tile_flux<1>(limiter, variant, false, T, in, out, wait_in, wait_out, eos, ctl, s);
}

}  // namespace zfv
