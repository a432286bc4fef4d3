// Instantiations and dispatch of the register-resident forward and inverse stage kernels.
// Compiled six times: as it stands for the stride permutation, and through ncn_fwd_indexed.hip (NCN_INDEXED_BUILD = 1)
// for launches that carry a grouping table or context lengths; each of the two takes every element type and activation
// and hands tanh launches of one storage type on to its builds for that type (ncn_fwd_f32.hip, ncn_fwd_bf16.hip,
// ncn_fwd_indexed_f32.hip, ncn_fwd_indexed_bf16.hip: NCN_TYPES_BUILD).
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
hipError_t launch_stage_forward<NCN_INDEXED_BUILD != 0, NCN_TYPES_BUILD>(Pass pass, const StageArgs& a, int grid_x, hipStream_t s) {
    constexpr bool kIndexed = NCN_INDEXED_BUILD != 0;
    constexpr int kTypes = NCN_TYPES_BUILD;
    const dim3 grid(grid_x), block(kBlockThreads);
    const bool tanh_only = a.activation == NCN_ACT_TANH;
    if constexpr (kTypes == kAnyTypes) {
        const int types = stage_types(pass, a);
        if (types == kF32Types) return launch_stage_forward<kIndexed, kF32Types>(pass, a, grid_x, s);
        if (types == kBf16Types) return launch_stage_forward<kIndexed, kBf16Types>(pass, a, grid_x, s);
    }
#define NCN_LAUNCH(KERNEL) hipLaunchKernelGGL(KERNEL, grid, block, 0, s, a)
#define NCN_CASE(NC, EC, R, F)                                                                        \
    static_assert(fast_tile(NC, EC).r == R && fast_tile(NC, EC).f == F, "duplicate config entry");    \
    if (a.n_cache == NC && a.head_dim == EC) {                                                        \
        if (tanh_only) {                                                                              \
            if (pass == kInverse) NCN_LAUNCH((stage_inverse_kernel<NC, EC, R, F, true, kIndexed, kTypes>));  \
            else NCN_LAUNCH((stage_forward_kernel<NC, EC, R, F, true, kIndexed, kTypes>));            \
        } else if constexpr (kTypes == kAnyTypes) {                                                   \
            if (pass == kInverse) NCN_LAUNCH((stage_inverse_kernel<NC, EC, R, F, false, kIndexed>));  \
            else NCN_LAUNCH((stage_forward_kernel<NC, EC, R, F, false, kIndexed>));                   \
        }                                                                                             \
        return hipGetLastError();                                                                     \
    }
    NCN_FOR_EACH_FAST_CONFIG(NCN_CASE)
#undef NCN_CASE
#undef NCN_LAUNCH
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
