// Instantiations and dispatch of the register-tile kernels for group sizes and head widths that are no powers of two.
// Compiled four times: as it stands (forward and inverse); through ncn_anyshape_bwd.hip (NCN_ANYSHAPE_BACKWARD = 1: the
// reversible backward); and each of the two once more for launches that carry context lengths
// (ncn_anyshape_lengths.hip, ncn_anyshape_bwd_lengths.hip: NCN_ANYSHAPE_LENGTHS = 1).
#include "ncn_anyshape_kernels.h"
#include "ncn_launch.h"

#ifndef NCN_ANYSHAPE_BACKWARD
#define NCN_ANYSHAPE_BACKWARD 0
#endif

#ifndef NCN_ANYSHAPE_LENGTHS
#define NCN_ANYSHAPE_LENGTHS 0
#endif

namespace ncn {

#define NCN_FOR_EACH_ANY_TILE(X) \
    X(2, 3) X(2, 4) X(2, 5) X(3, 3) X(3, 4) X(3, 5) X(4, 3) X(4, 4) X(4, 5) X(5, 3) X(5, 4) X(5, 5)

#if NCN_ANYSHAPE_BACKWARD && NCN_ANYSHAPE_LENGTHS
hipError_t launch_any_backward_lengths(const StageArgs& a, int grid_x, hipStream_t s) {
#elif NCN_ANYSHAPE_BACKWARD
hipError_t launch_any_backward(const StageArgs& a, int grid_x, hipStream_t s) {
    if (a.ctx_len) return launch_any_backward_lengths(a, grid_x, s);
#elif NCN_ANYSHAPE_LENGTHS
hipError_t launch_any_forward_lengths(Pass pass, const StageArgs& a, int grid_x, hipStream_t s) {
#else
hipError_t launch_any_forward(Pass pass, const StageArgs& a, int grid_x, hipStream_t s) {
    if (a.ctx_len) return launch_any_forward_lengths(pass, a, grid_x, s);
#endif
    constexpr bool kLengths = NCN_ANYSHAPE_LENGTHS != 0;
    const int r = a.any_tile & 0xff, f = (a.any_tile >> 8) & 0xff;
    const bool tanh_only = a.activation == NCN_ACT_TANH;
#define NCN_LAUNCH(KERNEL) hipLaunchKernelGGL(KERNEL, dim3(grid_x), dim3(kBlockThreads), 0, s, a)
#if NCN_ANYSHAPE_BACKWARD
    const bool loop = (uint64_t)a.total_tiles * (uint64_t)a.n_head > (uint64_t)grid_x * kWavesPerBlock;   // more tiles than waves
#define NCN_CASE(R, F)                                                                  \
    if (r == R && f == F) {                                                             \
        if constexpr (R * F <= 15) {                                                    \
            if (tanh_only && !loop) {                                                   \
                NCN_LAUNCH((any_backward_kernel<R, F, true, kLengths, false>));         \
                return hipGetLastError();                                               \
            }                                                                           \
        }                                                                               \
        if (tanh_only) NCN_LAUNCH((any_backward_kernel<R, F, true, kLengths, true>));        \
        else NCN_LAUNCH((any_backward_kernel<R, F, false, kLengths, true>));                      \
        return hipGetLastError();                                                       \
    }
#else
    const bool priority = tanh_only && !kLengths && a.n_cache >= kAnyPriorityRows;
#define NCN_CASE(R, F)                                                                  \
    if (r == R && f == F) {                                                             \
        if (pass == kInverse) {                                                         \
            if (priority) NCN_LAUNCH((any_forward_kernel<R, F, true, true, kLengths, !kLengths>)); \
            else if (tanh_only) NCN_LAUNCH((any_forward_kernel<R, F, true, true, kLengths, false>)); \
            else NCN_LAUNCH((any_forward_kernel<R, F, false, true, kLengths, false>));            \
        } else {                                                                        \
            if (priority) NCN_LAUNCH((any_forward_kernel<R, F, true, false, kLengths, !kLengths>)); \
            else if (tanh_only) NCN_LAUNCH((any_forward_kernel<R, F, true, false, kLengths, false>)); \
            else NCN_LAUNCH((any_forward_kernel<R, F, false, false, kLengths, false>));           \
        }                                                                               \
        return hipGetLastError();                                                       \
    }
#endif
    NCN_FOR_EACH_ANY_TILE(NCN_CASE)
#undef NCN_CASE
#undef NCN_LAUNCH
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
