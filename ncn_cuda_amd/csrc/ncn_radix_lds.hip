// Passes over radix-n levels of launches with few workgroups: the RADIX builds of the multi-stage kernels that keep their rows in
// LDS (ncn_fused_kernels.h), for heads of several features and (NCN_RADIX_HEADWISE) of one.  Planning and the choice between these
// and the kernels that keep them in registers: ncn_radix.hip.
#include "ncn_fused_dispatch.h"

#ifndef NCN_RADIX_HEADWISE
#define NCN_RADIX_HEADWISE false
#endif

namespace ncn {

template <>
hipError_t launch_radix_lds<NCN_RADIX_HEADWISE>(Pass pass, const FusedArgs& a, int nc, int ec, int grid, hipStream_t s) {
    const TileShape t = fast_tile(nc, ec);
    const bool backward = pass == kBackward;
    const int nw = backward ? kFusedWavesBwd : kFusedWavesFwd;
    size_t lds = ((size_t)(backward ? 4 : 2) * a.window * nc + 2 * kFusedMaxStages) * ec * sizeof(float);
    if (nc > t.r) lds += (size_t)nw * t.f * 64 * sizeof(float);
    if (backward) lds += (size_t)nw * a.n_stages * 2 * ec * sizeof(float);
    return launch_fused_shape<true, false, NCN_RADIX_HEADWISE>(pass, a, nc, ec, grid, lds, s);
}

}  // namespace ncn
