// Host-side launch interface between the C ABI (ncn_api.hip) and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "ncn_configs.h"
#include "ncn_device.h"

namespace ncn {

enum Pass { kForward = 0, kInverse = 1, kBackward = 2 };

// Register tile (rows x features per lane) the register kernels use for (n_cache, head width); {0,0} = none.
struct TileShape {
    int r, f;
};
constexpr TileShape fast_tile(int nc, int ec) {
#define NCN_MATCH(NC, EC, R, F) \
    if (nc == NC && ec == EC) return TileShape{R, F};
    NCN_FOR_EACH_FAST_CONFIG(NCN_MATCH)
#undef NCN_MATCH
    return TileShape{0, 0};
}

// Groups that one 64-lane wave tile carries on each path.
inline int fast_groups_per_tile(int nc, int ec) {
    const TileShape t = fast_tile(nc, ec);
    return 64 / ((nc / t.r) * (ec / t.f));
}
inline int generic_groups_per_tile(int nc) { return 64 / nc; }

// Largest head width the generic LDS kernel can hold (7 float arrays of [Ec][64] in 160 KB of LDS).
constexpr int kGenericMaxHeadDim = 64;
constexpr int kGenericArrays = 7;

// Upper bound on gridDim.x of a stage launch == rows of the dW partial buffer.
constexpr int kMaxGridX = 16384;
// Upper bound on gridDim.x of a forward / inverse launch (no partial rows to pay for).
constexpr int kMaxForwardGridX = 1 << 18;
// dW partial rows are summed in one launch where no segment has more than kReduceOneLaunchRows (ncn_generic.hip), else in two
// levels: chunks of kReduceRowsPerBlock rows, then the chunk sums.
constexpr int kReduceRowsPerBlock = 32;
// One reduction job sums up to kReduceMaxSegments partial arrays (one per backward launch of a call) that lie side by
// side in the partial buffer and hold at most kReduceMaxStages stages between them.
constexpr int kReduceMaxSegments = 8;
constexpr int kReduceMaxStages = 8;
// Rows of 2E floats that level 1 may need: sum over segments of ceil(rows / 32) * stages, where the segments' rows *
// stages add up to at most kMaxGridX and their stages to at most kReduceMaxStages.
constexpr int kReduceLevel1Rows = kMaxGridX / kReduceRowsPerBlock + kReduceMaxStages;
struct ReduceSegment {
    const float* in;        // [rows][cols], dense
    void* out;              // [cols] of the job's out_dtype
    int64_t cols;           // stages of the launch * 2E
    int64_t level1_offset;  // floats before this segment's chunk sums in the level-1 scratch
    int rows;
    int chunk0;             // chunks of the segments before this one
};
struct ReduceJob {
    ReduceSegment seg[kReduceMaxSegments];
    int n;
    int out_dtype;
};
// out[col] of every segment = sum of its rows, in a fixed order; level1 is scratch of kReduceLevel1Rows * 2E floats.
hipError_t launch_reduce_job(const ReduceJob& job, float* level1, hipStream_t s);

// Raises a kernel's dynamic LDS limit to `bytes` on the current device unless an earlier call already raised it that
// far (the limit is kept per device and kernel for the life of the process: one driver call instead of one per launch).
hipError_t ensure_dynamic_lds(const void* kernel, size_t bytes);

// Element types of a launch, where a kernel is built for one combination (tanh builds): with the branch on the type gone
// the loads of a tile go straight into its registers and nothing is copied where the branches meet.
//   kAnyTypes: read from the arguments
//   kAnyTypesOnce: the same in the backward, where the grid has a wave for every tile.  The build with a loop over tiles
//   needs more registers: relu, 16 x 2048 x 128, groups of 4, 36.8 us against 31.0 without the loop; tanh, 32 x 4096 x 128,
//   groups of 16, float32 outputs and bfloat16 gradients, 167.5 against 159.7
//   kF32Types: float32 everywhere
//   kBf16Types: bfloat16 storage -- forward and inverse read bfloat16, the backward reads saved outputs in two planes and
//   bfloat16 gradients, everything is written as bfloat16 (forward: one plane or two)
enum { kAnyTypes = -1, kF32Types = 0, kBf16Types = 1, kAnyTypesOnce = 2 };
// which of them a launch of the stage kernels is
inline int stage_types(Pass pass, const StageArgs& a) {
    if (a.activation != NCN_ACT_TANH) return kAnyTypes;
    if (a.in_dtype == NCN_F32 && a.out_dtype == NCN_F32 && (pass != kBackward || a.g_dtype == NCN_F32)) return kF32Types;
    const bool bf16 = pass == kForward    ? a.in_dtype == NCN_BF16 && a.out_dtype != NCN_F32
                      : pass == kInverse ? a.in_dtype == NCN_BF16 && a.out_dtype == NCN_BF16
                                         : a.in_dtype == NCN_BF16X2 && a.g_dtype == NCN_BF16 && a.out_dtype == NCN_BF16;
    return bf16 ? kBf16Types : kAnyTypes;
}
// One stage on the register kernels (ncn_fwd*.hip, ncn_bwd*.hip).  INDEXED: the builds that honour a.table,
// a.radix_stride and a.ctx_len.  Callers take TYPES = kAnyTypes, which goes to the other builds by itself.
template <bool INDEXED, int TYPES = kAnyTypes>
hipError_t launch_stage_forward(Pass pass, const StageArgs& a, int grid_x, hipStream_t s);
template <bool INDEXED, int TYPES = kAnyTypes>
hipError_t launch_stage_backward(const StageArgs& a, int grid_x, hipStream_t s);
#define NCN_DECLARE(INDEXED, TYPES)                                                                             \
    template <> hipError_t launch_stage_forward<INDEXED, TYPES>(Pass, const StageArgs&, int, hipStream_t);      \
    template <> hipError_t launch_stage_backward<INDEXED, TYPES>(const StageArgs&, int, hipStream_t);
NCN_DECLARE(false, kAnyTypes) NCN_DECLARE(false, kF32Types) NCN_DECLARE(false, kBf16Types)
NCN_DECLARE(true, kAnyTypes) NCN_DECLARE(true, kF32Types) NCN_DECLARE(true, kBf16Types)
#undef NCN_DECLARE
template <> hipError_t launch_stage_backward<false, kAnyTypesOnce>(const StageArgs&, int, hipStream_t);
template <> hipError_t launch_stage_backward<true, kAnyTypesOnce>(const StageArgs&, int, hipStream_t);
// Launches with few groups (ncn_split_kernels.h): tanh, one row fragment of 4 features per lane.
// The time of a launch here over that on the register tiles, float32, backward with its reduction (bfloat16 is within 0.05 of it but
// where named; behind a table):
//                 forward, 2^19   3 2^18   2^20 elements    backward, 2^19   3 2^18   2^20             tiles : here at 2^20, us
//   8 rows of  8      0.73  0.78  0.86 (table 0.83)            0.85  0.99  1.03 (table 0.97)            8.2 :  7.1, 14.1 : 14.6
//   8 rows of 16      0.75  0.81  0.90 (0.88)                  0.87  0.98  1.07 (1.04)                  7.6 :  6.8, 13.6 : 14.5
//   8 rows of 32      0.74  0.80  0.87 (0.85)                  0.80  0.91  1.00 (0.97)                  7.9 :  6.9, 14.8 : 14.8
//  16 rows of 16      0.72  0.80  0.93 (0.89)                  0.78  0.90  1.04 (1.00)                 10.3 :  9.6, 20.3 : 21.2
//  16 rows of 32      0.71  0.82  0.96 (0.90)                  0.77  0.86  1.01 (0.97)                 10.8 : 10.3, 22.7 : 22.9
//  32 rows of  4      0.58  0.72  0.82 (0.83)                  0.68  0.84  1.00, bfloat16 1.08 (0.93)
//  32 rows of 16      0.68  0.84  1.01 (0.95)                  0.79  0.91  1.09 (1.05)                 16.2 : 16.4, 35.1 : 38.2
//  32 rows of 32      0.67  0.81  0.98 (0.90)                  0.65  0.73  0.88 (0.84)                 17.0 : 16.8, 40.4 : 35.4
//  64 rows of  8      0.64  0.83  1.00 (0.99)                  0.71  0.85  1.03, bfloat16 1.07 (1.01)
//  64 rows of 16      0.65  0.87  1.03, bfloat16 1.12 (0.93)   0.67  0.78  0.96 (0.93)
// Heads of 64 and 128 (whose tiles hold 8 features per lane) and 64 rows of 32: at most 0.83 everywhere at 2^20.
// Smaller groups have short chains (their tile is 2 x 4).  Two rows, heads up to 32: forward 0.92 to 0.98 up to 2^17, 0.91 to 1.04 at
// 2^18, backward 0.91 to 1.02, 0.94 to 1.05; wider heads at most 0.97 at 2^18.  Four rows, 2^18: at most 0.98; 2^19: up to 1.08.
constexpr int64_t split_max_elements(int n_cache, int head_dim, bool backward, bool indexed) {
    if (n_cache == 2) return head_dim <= 32 ? 1 << 17 : 1 << 18;
    if (n_cache == 4) return 1 << 18;
    const bool even_earlier = backward ? (head_dim == 16 && n_cache <= 32) || (head_dim == 8 && (n_cache == 8 || n_cache == 64)) ||
                                             (head_dim == 4 && n_cache == 32)
                                       : (head_dim == 16 && n_cache >= 32) || (head_dim == 8 && n_cache == 64);
    return !indexed && even_earlier ? 3 << 18 : 1 << 20;
}
int split_groups_per_tile(int nc, int ec);
// indexed: the builds that honour a.table, a.radix_stride and a.ctx_len
hipError_t launch_split(Pass pass, const StageArgs& a, bool indexed, hipStream_t s);
// Heads of one feature (ncn_headwise_kernels.h): `a` carries the geometry of E / w heads of w features, w =
// headwise_width(E), for which the grid was planned as well; the second form honours a.table, a.radix_stride and
// a.ctx_len.
constexpr int kHeadwiseMaxWidth = 32;
// adjacent one-feature heads that the lanes of a row hold together: the largest of 32, 16, 8, 4 that divides E (0: none)
constexpr int headwise_width(int64_t E) {
    for (int w = kHeadwiseMaxWidth; w >= 4; w /= 2)
        if (E % w == 0) return w;
    return 0;
}
hipError_t launch_headwise_forward(Pass pass, const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_headwise_forward_indexed(Pass pass, const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_headwise_backward(const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_headwise_backward_indexed(const StageArgs& a, int grid_x, hipStream_t s);
// Shapes that are no powers of two (ncn_anyshape_kernels.h): a.any_tile says which tile.
struct AnyTile {
    int r, f;               // rows and features per lane; r == 0: no tile holds the group in one wave
    int lf_log2, lr_log2;   // log2 of the lanes per row and of the row lanes per group
};
// The tile whose wave issues the least for a group: padded elements times what one costs (some 20 instructions), plus
// the sums across lanes (2 R over the lanes of a row, F over the row lanes) and the pivot row's own terms, per lane.  Tiles
// of more than 16 elements (two or three waves per SIMD) only where the group fits no smaller one.
inline AnyTile any_tile(int nc, int ec) {
    AnyTile best{0, 0, 0, 0};
    int best_cost = 0;
    for (int r = 2; r <= 5; ++r)
        for (int f = 3; f <= 5; ++f) {
            int lf = 0, lr = 0;
            while ((f << lf) < ec) ++lf;
            while ((r << lr) < nc) ++lr;
            if (lf + lr > 6 || lf > 5) continue;
            int cost = (20 * r * f + 4 * r * lf + 2 * f * lr + 10 * f) << (lf + lr);
            if (r * f > 16) cost *= 4;
            if (best.r == 0 || cost < best_cost) {
                best = AnyTile{r, f, lf, lr};
                best_cost = cost;
            }
        }
    return best;
}
hipError_t launch_any_forward(Pass pass, const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_any_backward(const StageArgs& a, int grid_x, hipStream_t s);
// the builds with context lengths (a.ctx_len set); the two above go there by themselves
hipError_t launch_any_forward_lengths(Pass pass, const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_any_backward_lengths(const StageArgs& a, int grid_x, hipStream_t s);
hipError_t launch_generic(Pass pass, const StageArgs& a, int n_head, int grid_x, hipStream_t s);
// Rows past the context length of their batch entry: copied through (a.ctx_len must be set).
hipError_t launch_pass_through(Pass pass, const StageArgs& a, int64_t batch, hipStream_t s);
// gridDim.x of the generic kernel's edge launch (the partly live group of each batch entry) == its dW partial rows.
constexpr int kEdgeGridX = 256;
// ---- multi-stage (LDS-resident) passes, ncn_fused.hip --------------------------------------------------------
struct FusedArgs;
struct FusedPass {
    int first, count;  // stages [first, first + count) relative to the range that was planned
    int single;        // 1: not worth fusing, run `first` with the one-stage kernel
    uint32_t class_stride, ring, window, halo, own, tiles_per_ring, closed, class_groups;
    uint32_t sub_stride[8];
    // halo pass: what slot 1 has moved against its place at the pass's first stage, and the groups that the windows need in front
    // of and behind the owned ones when the stages run in ascending order (the other way round in descending order)
    int32_t shear[8];
    uint32_t before, after;
};
bool fused_supported(const ncn_shape* sh, int activation);
// sheared = false: the cuts that ncn_plan_passes reports
std::vector<FusedPass> plan_fused(const ncn_shape* sh, int first, int count, bool backward, bool sheared = false);
// Consecutive stages of a trained stack whose last outputs are kept for the backward: the passes of both directions, in
// ascending order, numbered relative to the planned stages.
struct StackRange {
    std::vector<FusedPass> fwd, bwd;
};
// At most max_saves ranges of at most max_range stages, both at most `count` (empty if there is no such cut).  multi_stage: whether the shape has
// multi-stage passes; without them every pass is one stage.
std::vector<StackRange> plan_stack(const ncn_shape* sh, int first, int count, bool multi_stage, int max_range, int max_saves);
// windows of a pass (== workgroups, when every workgroup takes one)
int64_t fused_items(const ncn_shape* sh, const FusedPass& p);
// workgroups of a backward pass.  row_cap: rows of the dW partial buffer it may fill (grid / n_head rows per stage)
int fused_backward_grid(const ncn_shape* sh, const FusedPass& p, int row_cap);
// row_cap: as above
// headwise: `sh` is the layout of a call on heads of one feature (headwise_width(E) adjacent heads to a "head")
hipError_t launch_fused(Pass pass, FusedArgs& a, const ncn_shape* sh, const FusedPass& p, hipStream_t s,
                        int row_cap = kMaxGridX, bool headwise = false);
// the builds with context lengths (a.ctx_len set), ncn_fused_lengths.hip; launch_fused goes there by itself
hipError_t launch_fused_lengths(Pass pass, const FusedArgs& a, int nc, int ec, int grid, size_t lds, hipStream_t s);
// the builds for heads of one feature (ncn_fused_headwise.hip; the first goes to the second when a.ctx_len is set)
hipError_t launch_fused_headwise(Pass pass, const FusedArgs& a, int nc, int ec, int grid, size_t lds, hipStream_t s);
hipError_t launch_fused_headwise_lengths(Pass pass, const FusedArgs& a, int nc, int ec, int grid, size_t lds, hipStream_t s);


// ---- multi-stage passes over radix-n levels, ncn_radix.hip ---------------------------------------------
struct RadixPass {
    int first, count;  // levels [first, first + count) relative to the range that was planned
    int single;        // 1: one level, run with the one-stage kernel
    uint32_t s0;       // n^(first level of the pass): distance in rows between the rows of a window
    uint32_t span;     // n^count: rows of a window
    uint32_t rows;     // rows of one batch entry that a workgroup holds (a whole number of windows)
    uint32_t loads;    // workgroup-loads per batch entry and head, when it holds no others
};
bool radix_fused_supported(const ncn_shape* sh);
// fused = false: one level per pass whatever the shape (calls whose scalars only the generic kernels take)
std::vector<RadixPass> plan_radix(const ncn_shape* sh, int first, int count, bool backward, bool fused = true);
int radix_grid(const ncn_shape* sh, const RadixPass& p, bool backward, bool tanh);
hipError_t launch_fused_radix(Pass pass, FusedArgs& a, const ncn_shape* sh, const RadixPass& p, hipStream_t s,
                              bool headwise = false);
// the builds that keep rows in LDS, heads of several features or of one (ncn_radix_lds.hip)
template <bool HEADWISE>
hipError_t launch_radix_lds(Pass pass, const FusedArgs& a, int nc, int ec, int grid, hipStream_t s);
template <> hipError_t launch_radix_lds<false>(Pass, const FusedArgs&, int, int, int, hipStream_t);
template <> hipError_t launch_radix_lds<true>(Pass, const FusedArgs&, int, int, int, hipStream_t);
// those that keep them in registers, by kind (ncn_radix_build.hip and the units that include it)
template <bool HEADWISE, bool BACKWARD, bool TANH>
hipError_t launch_radix(Pass pass, const FusedArgs& a, int nc, int ec, int grid, hipStream_t s);
#define NCN_DECLARE(H, B) \
    template <> hipError_t launch_radix<H, B, true>(Pass, const FusedArgs&, int, int, int, hipStream_t); \
    template <> hipError_t launch_radix<H, B, false>(Pass, const FusedArgs&, int, int, int, hipStream_t);
NCN_DECLARE(false, false) NCN_DECLARE(false, true) NCN_DECLARE(true, false) NCN_DECLARE(true, true)
#undef NCN_DECLARE

}  // namespace ncn
