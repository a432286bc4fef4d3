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

// Rows that a workgroup holds: its kernels keep them in registers (RadixShape::T bits of them)
uint32_t capacity_rows(int ec, bool backward) {
    return floor_pow2((uint32_t)(fused_state_bytes(backward) / ((backward ? 4 : 2) * ec * sizeof(float))));
}

// The workgroup-loads of a pass per head.  Windows of one batch entry (p.rows) leave a workgroup partly empty where their number
// has no divisor that fills it; counted through all entries they need fewer workgroups, each of which takes the same time.
struct RadixLoads {
    uint32_t rows;     // per workgroup
    int64_t loads;
    bool across;       // .. of windows counted through all batch entries
};
RadixLoads radix_loads(const ncn_shape* sh, const RadixPass& p, bool backward) {
    const uint32_t cap = capacity_rows((int)(sh->E / sh->n_head), backward);
    const int64_t whole = sh->batch * (int64_t)p.loads, per = cap / p.span;
    const int64_t across = (sh->batch * (sh->N / p.span) + per - 1) / per;
    if (across < whole) return RadixLoads{cap, across, true};
    return RadixLoads{p.rows, whole, false};
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

// Levels [first, first + count) cut into passes of as many levels as a workgroup's rows take (and the stage limits of the
// kernels); a pass of one level is left to the one-stage kernel.  Every pass is closed.
std::vector<RadixPass> plan_radix(const ncn_shape* sh, int first, int count, bool backward, bool fused) {
    std::vector<RadixPass> passes;
    const int nc = sh->n_cache, ec = (int)(sh->E / sh->n_head);
    const uint32_t cap_rows = capacity_rows(ec, backward);
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
        // A workgroup holds a whole number of windows, and every workgroup-load of a batch entry the same number: the largest
        // divisor of the window count that it takes (N = odd * n^k leaves an odd factor in the window count).
        const uint32_t windows = (uint32_t)(sh->N / p.span);   // per batch entry and head
        uint32_t per_load = cap_rows / p.span;
        if (per_load > windows) per_load = windows;            // N smaller than a workgroup
        while (windows % per_load) --per_load;
        p.rows = per_load * p.span;
        p.loads = windows / per_load;
        passes.push_back(p);
        a += p.count;
    }
    return passes;
}

int radix_grid(const ncn_shape* sh, const RadixPass& p, bool backward) {
    const int64_t items = radix_loads(sh, p, backward).loads * sh->n_head;
    // a workgroup for every item: filled ones need more than the card's memory before they exceed a grid
    if (!backward) return items <= INT_MAX ? (int)items : 0;
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
    const RadixLoads l = radix_loads(sh, p, backward);
    const int64_t windows = sh->N / p.span, per = l.rows / p.span;
    a.window = l.rows / nc;
    a.class_groups = l.across ? 0 : p.loads;
    a.entry_windows = (uint32_t)windows;
    a.entry_magic = windows < per ? (uint32_t)(((1ull << 31) + windows - 1) / windows) : 0;   // (exact: window numbers < 2 per)
    a.all_windows = (uint32_t)(sh->batch * windows);
    a.total_items = (uint32_t)(l.loads * sh->n_head);
    a.scale_dn = (float)std::pow((double)a.tab.m, (double)(nc * p.count));
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
