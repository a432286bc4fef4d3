// Instantiations and dispatch of the one-stage kernels for launches with few groups (ncn_split_kernels.h).
#include "ncn_configs.h"
#include "ncn_launch.h"
#include "ncn_split_kernels.h"

namespace ncn {

int split_groups_per_tile(int nc, int ec) {
    const int rows = 64 / (ec / 4);
    return nc > rows ? 1 : rows / nc;
}

template <bool INDEXED>
static hipError_t launch_split_build(Pass pass, const StageArgs& a, hipStream_t s) {
    const uint64_t units = (uint64_t)a.total_tiles * (uint64_t)a.n_head;
#define NCN_CASE(NC, EC, R, F)                                                                               \
    if (a.n_cache == NC && a.head_dim == EC) {                                                               \
        using S = SplitShape<NC, EC>;                                                                        \
        const dim3 grid((uint32_t)((units + S::UNITS - 1) / S::UNITS)), block(64 * S::NW);                   \
        if (pass == kBackward) hipLaunchKernelGGL((split_backward_kernel<NC, EC, INDEXED>), grid, block, 0, s, a);    \
        else if (pass == kInverse) hipLaunchKernelGGL((split_forward_kernel<NC, EC, true, INDEXED>), grid, block, 0, s, a); \
        else hipLaunchKernelGGL((split_forward_kernel<NC, EC, false, INDEXED>), grid, block, 0, s, a);       \
        return hipGetLastError();                                                                            \
    }
    NCN_FOR_EACH_FAST_CONFIG(NCN_CASE)
#undef NCN_CASE
    return hipErrorInvalidConfiguration;
}

hipError_t launch_split(Pass pass, const StageArgs& a, bool indexed, hipStream_t s) {
    return indexed ? launch_split_build<true>(pass, a, s) : launch_split_build<false>(pass, a, s);
}

}  // namespace ncn
