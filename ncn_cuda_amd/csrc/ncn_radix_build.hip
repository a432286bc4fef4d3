// Instantiations and dispatch of the radix kernels (ncn_radix_kernels.h): compiled eight times, for forward and inverse or
// backward, tanh or every activation, heads of several features or of one (NCN_RADIX_BACKWARD, _TANH, _HEADWISE); as it stands
// forward and inverse of tanh on heads of several features.
#include "ncn_launch.h"
#include "ncn_radix_kernels.h"

#ifndef NCN_RADIX_BACKWARD
#define NCN_RADIX_BACKWARD false
#endif
#ifndef NCN_RADIX_TANH
#define NCN_RADIX_TANH true
#endif
#ifndef NCN_RADIX_HEADWISE
#define NCN_RADIX_HEADWISE false
#endif

namespace ncn {

namespace {

template <int NC, int EC>
hipError_t launch_radix_shape(Pass pass, const FusedArgs& a, int grid, hipStream_t s) {
    constexpr bool kTanh = NCN_RADIX_TANH, kHeadwise = NCN_RADIX_HEADWISE;
    using S = RadixShape<NC, EC, NCN_RADIX_BACKWARD>;
    // what plan_radix gives a workgroup is what it holds: all slots, and levels on whole digits of their bits
    static_assert(((size_t)EC * sizeof(float) << S::T) * (NCN_RADIX_BACKWARD ? 4 : 2) == fused_state_bytes(NCN_RADIX_BACKWARD), "rows of a workgroup");
    if (a.window * NC > (1u << S::T) || a.n_stages * S::DB > S::TU) return hipErrorInvalidConfiguration;
    const bool loop = (uint32_t)grid < a.total_items;
    void (*k)(const FusedArgs);
    size_t lds = (size_t)kFusedMaxStages * 2 * EC * sizeof(float) + ((size_t)EC * sizeof(float) << S::T);
    if constexpr (NCN_RADIX_BACKWARD) {
        // (the looping build serves every launch of the other activations)
        if constexpr (kTanh) k = loop ? radix_backward_kernel<NC, EC, true, true, kHeadwise> : radix_backward_kernel<NC, EC, true, false, kHeadwise>;
        else k = radix_backward_kernel<NC, EC, false, true, kHeadwise>;
        lds += (size_t)S::NW * a.n_stages * 2 * EC * sizeof(float);
    } else {
        if (loop) return hipErrorInvalidConfiguration;   // a workgroup for every item
        k = pass == kInverse ? radix_forward_kernel<NC, EC, kTanh, true, kHeadwise> : radix_forward_kernel<NC, EC, kTanh, false, kHeadwise>;
    }
    const hipError_t err = ensure_dynamic_lds(reinterpret_cast<const void*>(k), lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k, dim3(grid), dim3(64 * S::NW), lds, s, a);
    return hipGetLastError();
}

}  // namespace

template <>
hipError_t launch_radix<NCN_RADIX_HEADWISE, NCN_RADIX_BACKWARD, NCN_RADIX_TANH>(Pass pass, const FusedArgs& a, int nc, int ec, int grid,
                                                                              hipStream_t s) {
    // one-feature heads are laid out as heads of up to kHeadwiseMaxWidth of them
#define NCN_CASE(NC, EC)                                                                                  \
    if constexpr (!NCN_RADIX_HEADWISE || EC <= kHeadwiseMaxWidth) {                                       \
        if (nc == NC && ec == EC) return launch_radix_shape<NC, EC>(pass, a, grid, s);                    \
    }
    NCN_FOR_EACH_FUSED_CONFIG(NCN_CASE)
#undef NCN_CASE
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
