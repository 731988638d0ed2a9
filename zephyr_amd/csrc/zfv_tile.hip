// The tiled steps' launchers; HLLC's MUSCL kernels (zfv_tile.hpp) and the
// first-order ones.  HLL's and Rusanov's are compiled in zfv_tile_flux.hip.
#include "zfv_tile.hpp"

namespace zfv {

hipError_t launch_tile_hll(int limiter, int variant, const TileMesh& T, const DevState& in, const DevState& out,
                           const int* wait_in, int* wait_out, const Eos& eos, const StepCtl& ctl, hipStream_t s);
hipError_t launch_tile_rusanov(int limiter, int variant, const TileMesh& T, const DevState& in, const DevState& out,
                               const int* wait_in, int* wait_out, const Eos& eos, const StepCtl& ctl, hipStream_t s);

bool tile_flux_built(int flux) { return flux >= 1 && flux <= 3; }

hipError_t launch_tile_step(int flux, int limiter, int variant, bool persistent, const TileMesh& T,
                            const DevState& in, const DevState& out, const int* wait_in, int* wait_out,
                            const Eos& eos, const StepCtl& ctl, hipStream_t s) {
    if (variant < 0 || variant >= kTileVariants || !tile_flux_built(flux)) return hipErrorInvalidValue;
    if (T.n_tiles[variant] <= 0) return hipSuccess;
    switch (flux) {
        case 1: return launch_tile_rusanov(limiter, variant, T, in, out, wait_in, wait_out, eos, ctl, s);
        case 2: return launch_tile_hll(limiter, variant, T, in, out, wait_in, wait_out, eos, ctl, s);
        default:
            return launch_tile_flux<3>(limiter, variant, persistent, T, in, out, wait_in, wait_out, eos, ctl, s);
    }
}

template <int V>
static hipError_t launch_tile_flux1_t(int flux, const TileMesh& T, const DevState& in, const DevState& out,
                                      const Eos& eos, const StepCtl& ctl, hipStream_t s) {
    constexpr int TI = kTileRows[V];
    const dim3 g(T.n_tiles[V]), b((TI + 2) * 64);
    switch (flux) {
        case 1: hipLaunchKernelGGL((k_tile_flux1<1, V, TI>), g, b, 0, s, T, in, out, eos, ctl); break;
        case 2: hipLaunchKernelGGL((k_tile_flux1<2, V, TI>), g, b, 0, s, T, in, out, eos, ctl); break;
        default: hipLaunchKernelGGL((k_tile_flux1<3, V, TI>), g, b, 0, s, T, in, out, eos, ctl); break;
    }
    return hipGetLastError();
}

hipError_t launch_tile_flux1(int flux, int variant, const TileMesh& T, const DevState& in, const DevState& out,
                             const Eos& eos, const StepCtl& ctl, hipStream_t s) {
    if (variant < 0 || variant >= kTileVariants || !tile_flux_built(flux)) return hipErrorInvalidValue;
    if (T.n_tiles[variant] <= 0) return hipSuccess;
    switch (variant) {
        case 0: return launch_tile_flux1_t<0>(flux, T, in, out, eos, ctl, s);
        case 1: return launch_tile_flux1_t<1>(flux, T, in, out, eos, ctl, s);
        case 2: return launch_tile_flux1_t<2>(flux, T, in, out, eos, ctl, s);
        default: return launch_tile_flux1_t<3>(flux, T, in, out, eos, ctl, s);
    }
}

}  // namespace zfv
