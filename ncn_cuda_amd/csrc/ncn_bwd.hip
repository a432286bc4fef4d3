// Instantiations and dispatch of the register-resident reversible backward stage kernel.
// Compiled eight times: as it stands for the stride permutation, and through ncn_bwd_indexed.hip (NCN_INDEXED_BUILD = 1)
// for launches that carry a grouping table or context lengths; each of the two takes every element type and activation,
// with a loop over tiles, and hands launches whose grid has a wave for every tile on to its builds without the loop
// (NCN_TYPES_BUILD): tanh of one storage type to ncn_bwd_f32.hip, ncn_bwd_bf16.hip, ncn_bwd_indexed_f32.hip and
// ncn_bwd_indexed_bf16.hip, everything else to ncn_bwd_once.hip and ncn_bwd_indexed_once.hip.
#include "ncn_configs.h"
#include "ncn_launch.h"
#include "ncn_stage_kernels.h"

#ifndef NCN_INDEXED_BUILD
#define NCN_INDEXED_BUILD 0
#endif
#ifndef NCN_TYPES_BUILD
#define NCN_TYPES_BUILD kAnyTypes
#endif

namespace ncn {

template <>
hipError_t launch_stage_backward<NCN_INDEXED_BUILD != 0, NCN_TYPES_BUILD>(const StageArgs& a, int grid_x, hipStream_t s) {
    constexpr bool kIndexed = NCN_INDEXED_BUILD != 0;
    constexpr bool kLoop = NCN_TYPES_BUILD == kAnyTypes;
    constexpr int kTypes = NCN_TYPES_BUILD == kAnyTypesOnce ? kAnyTypes : NCN_TYPES_BUILD;
    const dim3 grid(grid_x), block(kBlockThreads);
    const bool tanh_only = a.activation == NCN_ACT_TANH;
    if constexpr (kLoop) {
        if ((uint64_t)a.total_tiles * (uint64_t)a.n_head <= (uint64_t)grid_x * kWavesPerBlock) {   // a wave for every tile
            const int types = stage_types(kBackward, a);
            if (types == kF32Types) return launch_stage_backward<kIndexed, kF32Types>(a, grid_x, s);
            if (types == kBf16Types) return launch_stage_backward<kIndexed, kBf16Types>(a, grid_x, s);
            return launch_stage_backward<kIndexed, kAnyTypesOnce>(a, grid_x, s);
        }
    }
#define NCN_LAUNCH(KERNEL) hipLaunchKernelGGL(KERNEL, grid, block, 0, s, a)
#define NCN_CASE(NC, EC, R, F)                                                                        \
    static_assert(fast_tile(NC, EC).r == R && fast_tile(NC, EC).f == F, "duplicate config entry");    \
    if (a.n_cache == NC && a.head_dim == EC) {                                                        \
        if (tanh_only) NCN_LAUNCH((stage_backward_kernel<NC, EC, R, F, true, kIndexed, kLoop, kTypes>));     \
        else if constexpr (kTypes == kAnyTypes) NCN_LAUNCH((stage_backward_kernel<NC, EC, R, F, false, kIndexed, kLoop>)); \
        return hipGetLastError();                                                                     \
    }
    NCN_FOR_EACH_FAST_CONFIG(NCN_CASE)
#undef NCN_CASE
#undef NCN_LAUNCH
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
