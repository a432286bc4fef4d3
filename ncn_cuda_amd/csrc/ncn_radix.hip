// Planning and launching of multi-stage passes over levels of the radix-n digit grouping
// (ncn_triton/group_tensors.py:8-18); the kernels are those of ncn_radix_kernels.h,
// built in ncn_radix_build.hip.
#include <climits>
#include <cmath>
#include <vector>

#include "ncn_configs.h"
#include "ncn_fused_kernels.h"
#include "ncn_launch.h"

namespace ncn {

namespace {

// shapes with a radix build: digits are bits of a row number, so n_cache is 2 or 4
#define NCN_FOR_EACH_RADIX_CONFIG(X) NCN_FOR_EACH_FUSED_CONFIG(X)

uint32_t floor_pow2(uint32_t v) {
    uint32_t p = 1;
    while (p * 2 <= v) p *= 2;
    return p;
}

int64_t ipow(int64_t b, int e) {
    int64_t r = 1;
    for (int k = 0; k < e; ++k) r *= b;
    return r;
}

}  // namespace

bool radix_fused_supported(const ncn_shape* sh) {
    const int64_t ec = sh->E / sh->n_head;
#define NCN_MATCH(NC, EC) \
    if (sh->n_cache == NC && ec == EC) return true;
    NCN_FOR_EACH_RADIX_CONFIG(NCN_MATCH)
#undef NCN_MATCH
    return false;
}

// Levels [first, first + count) cut into passes of as many levels as fit the LDS budget (and the stage limits of the
// kernels); a pass of one level is left to the one-stage kernel.  Every pass is closed.
std::vector<RadixPass> plan_radix(const ncn_shape* sh, int first, int count, bool backward, bool fused) {
    std::vector<RadixPass> passes;
    const int nc = sh->n_cache, ec = (int)(sh->E / sh->n_head);
    const uint32_t cap_rows = floor_pow2((uint32_t)(fused_state_bytes(backward) / ((backward ? 4 : 2) * ec * sizeof(float))));
    int kmax = 0;
    while (ipow(nc, kmax + 1) <= (int64_t)cap_rows) ++kmax;
    const int max_stages = backward ? kFusedMaxStages - 1 : kFusedMaxStages;
    if (kmax > max_stages) kmax = max_stages;
    for (int a = 0; a < count;) {
        RadixPass p{};
        p.first = a;
        p.count = (count - a < kmax) ? count - a : kmax;
        p.single = (p.count < 2 || !fused || !radix_fused_supported(sh)) ? 1 : 0;
        if (p.single) p.count = 1;
        p.s0 = (uint32_t)ipow(nc, first + a);
        p.span = (uint32_t)ipow(nc, p.count);
        // A workgroup holds a whole number of windows, and every workgroup-load of a batch entry holds the same
        // number: the largest divisor of the window count that the LDS budget takes (N = odd * n^k leaves an odd
        // factor in the window count; a count that does not divide would leave the last windows unprocessed).
        const uint32_t windows = (uint32_t)(sh->N / p.span);   // per batch entry and head
        uint32_t per_load = cap_rows / p.span;
        if (per_load > windows) per_load = windows;            // N smaller than the LDS budget
        while (windows % per_load) --per_load;
        p.rows = per_load * p.span;
        p.loads = windows / per_load;
        passes.push_back(p);
        a += p.count;
    }
    return passes;
}

int radix_grid(const ncn_shape* sh, const RadixPass& p, bool backward) {
    const int64_t items = sh->batch * (int64_t)p.loads * sh->n_head;
    if (!backward) return items <= INT_MAX ? (int)items : 0;   // a workgroup for every item
    // .. in the backward where the dW scratch has a partial row for each
    const int64_t by_rows = (int64_t)kMaxGridX / p.count * sh->n_head;
    int64_t g = items < by_rows ? items : by_rows;
    g = g / sh->n_head * sh->n_head;
    if (g < sh->n_head) g = sh->n_head;
    return (int)g;
}

hipError_t launch_fused_radix(Pass pass, FusedArgs& a, const ncn_shape* sh, const RadixPass& p, hipStream_t s,
                              bool headwise) {
    const bool backward = pass == kBackward;
    const int nc = sh->n_cache, ec = (int)(sh->E / sh->n_head);
    a.N = sh->N;
    a.E = sh->E;
    a.n_head = sh->n_head;
    a.n_stages = p.count;
    a.class_stride = p.s0;
    a.ring = p.span;
    a.window = p.rows / nc;
    a.halo = 0;
    a.own = a.window;
    a.tiles_per_ring = 1;
    a.closed = 1;
    a.class_groups = p.loads;
    a.total_items = (uint32_t)(sh->batch * (int64_t)p.loads * sh->n_head);
    for (int k = 0; k < kFusedMaxStages; ++k) a.sub_stride[k] = k < p.count ? (uint32_t)ipow(nc, k) : 0;
    a.scale_dn = (float)std::pow((double)a.tab.m, (double)(nc * p.count));
    a.scale_up = (float)std::pow((double)a.tab.m, -(double)(nc * p.count));
    const int grid = radix_grid(sh, p, backward);
    const bool tanh_only = a.tab.activation == NCN_ACT_TANH;
#define NCN_PICK(HEADWISE, BACKWARD, TANH) \
    if (headwise == HEADWISE && backward == BACKWARD && tanh_only == TANH) return launch_radix<HEADWISE, BACKWARD, TANH>(pass, a, nc, ec, grid, s);
    NCN_PICK(false, false, true) NCN_PICK(false, true, true) NCN_PICK(false, false, false) NCN_PICK(false, true, false)
    NCN_PICK(true, false, true) NCN_PICK(true, true, true) NCN_PICK(true, false, false) NCN_PICK(true, true, false)
#undef NCN_PICK
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
