// Planning and launching of multi-stage passes over levels of the radix-n digit grouping
// (ncn_triton/group_tensors.py:8-18); the kernels are those of ncn_radix_kernels.h, built in ncn_radix_build.hip, and in
// launches with few workgroups the RADIX builds of ncn_fused_kernels.h (ncn_radix_lds.hip).
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
    bool lds;          // for the kernels that keep rows in LDS
};

// Whether a launch of so many workgroups, of `rows` rows each, runs on the kernels that keep rows in LDS.  A lane of the register
// kernels holds 16 elements and more, and a workgroup takes the same time however few of its rows exist; the LDS kernels spread the
// rows there are over 8 waves, 8 elements to a lane, which is the shorter chain as long as every workgroup starts at once and has
// at most half the rows that fit.  tanh, us, LDS : registers, forward | backward, N = rows, by workgroups:
//   groups of two, heads of  8,  8 rows, 3 levels  64:  6.0 : 11.0 | 11.0 : 12.6   256:  6.1 : 11.4 | 11.3 : 12.9   512:  8.1 : 11.8 | 12.8 : 12.9
//   groups of two, heads of 32,  8 rows, 3 levels  64:  5.9 :  9.4 | 10.7 : 10.9   256:  6.0 :  9.5 | 10.9 : 11.2   512:  7.4 :  9.6 | 12.1 : 11.3
//   groups of two, heads of 32, 128 rows, 7 levels 64: 11.9 : 15.8 | 22.1 : 18.1   256: 13.1 : 16.8 | 24.0 : 19.6   512: 20.2 : 19.4 | 36.7 : 32.3
//   groups of two, heads of 64,  8 rows, 3 levels  64:  7.1 :  9.4 | 13.9 : 11.4   256:  7.3 :  9.5 | 14.3 : 11.6   512: 12.6 :  9.7 | 24.3 : 12.0
//   groups of four, heads of 32, 64 rows, 3 levels 64:  8.2 : 12.9 | 14.3 : 16.4   256:  8.8 : 13.4 | 15.2 : 17.3   512: 11.9 : 14.0 | 19.8 : 18.3
// With all the rows that fit (groups of two, heads of 16, 8 levels of 512 rows forward and 256 backward) registers win from the
// first workgroup on, by 10 and 11 %.
//   The other activations spend more instructions on an element, which 8 waves of few elements overlap better: the time on registers
// over that in LDS, relu, groups of two, by workgroups (512, 2048, 6000 unless named), forward heads of 16: 128 rows of 512 2.12, 0.78,
// 0.59, 256 rows 1.97, 1.23, 0.99, all 512 rows 1.27, 1.12, 1.07 (sigmoid 1.14, 1.03, 0.95); heads of 64: 64: 1.38, 256: 1.36, 512:
// 0.86; groups of four, heads of 8: 512 of 1024 rows 1.23, 0.82, 0.82, all of them 0.80.  Backward, heads of 32, all 128 rows: 64:
// 1.28, 256: 1.24, 512: 0.77; heads of 64 0.87 at 64.
bool rows_in_lds(int nc, int ec, bool backward, bool tanh, uint32_t rows, uint32_t cap, int64_t workgroups) {
    const bool half = 2 * rows <= cap, quarter = 4 * rows <= cap;
    if (tanh) {
        if (!half) return false;
        if (backward) return workgroups <= 256 && (ec <= 16 || (ec <= 32 && nc == 4));
        return workgroups <= (ec <= 16 || (ec <= 32 && quarter) ? 512 : 256);
    }
    if (backward) return workgroups <= 256 && ec <= 32;
    if (ec > 32) return workgroups <= 256;
    if (nc == 4 && ec == 8 && !quarter) return half && workgroups <= 512;
    return workgroups <= (quarter ? 512 : half ? 2048 : 4096);
}

RadixLoads radix_loads(const ncn_shape* sh, const RadixPass& p, bool backward, bool tanh) {
    const uint32_t cap = capacity_rows((int)(sh->E / sh->n_head), backward);
    const int64_t whole = sh->batch * (int64_t)p.loads, per = cap / p.span;
    const int64_t across = (sh->batch * (sh->N / p.span) + per - 1) / per;
    if (rows_in_lds(sh->n_cache, (int)(sh->E / sh->n_head), backward, tanh, p.rows, cap, whole * sh->n_head))
        return RadixLoads{p.rows, whole, false, true};
    if (across < whole) return RadixLoads{cap, across, true, false};
    return RadixLoads{p.rows, whole, false, false};
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

int radix_grid(const ncn_shape* sh, const RadixPass& p, bool backward, bool tanh) {
    const int64_t items = radix_loads(sh, p, backward, tanh).loads * sh->n_head;
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
    const bool tanh = a.tab.activation == NCN_ACT_TANH;
    const RadixLoads l = radix_loads(sh, p, backward, tanh);
    const int grid = radix_grid(sh, p, backward, tanh);
    const int64_t windows = sh->N / p.span, per = l.rows / p.span;
    a.window = l.rows / nc;
    a.class_groups = l.across ? 0 : p.loads;
    a.entry_windows = (uint32_t)windows;
    a.entry_magic = windows < per ? (uint32_t)(((1ull << 31) + windows - 1) / windows) : 0;   // (exact: window numbers < 2 per)
    a.all_windows = (uint32_t)(sh->batch * windows);
    a.total_items = (uint32_t)(l.loads * sh->n_head);
    a.scale_dn = (float)std::pow((double)a.tab.m, (double)(nc * p.count));
    if (l.lds) {
        a.own = a.window;
        a.tiles_per_ring = 1;
        a.closed = 1;
        for (int k = 0; k < p.count; ++k) a.sub_stride[k] = (uint32_t)ipow(nc, k);
        a.scale_up = (float)std::pow((double)a.tab.m, -(double)(nc * p.count));
        return headwise ? launch_radix_lds<true>(pass, a, nc, ec, grid, s) : launch_radix_lds<false>(pass, a, nc, ec, grid, s);
    }
#define NCN_PICK(HEADWISE, BACKWARD, TANH) \
    if (headwise == HEADWISE && backward == BACKWARD && tanh == TANH) return launch_radix<HEADWISE, BACKWARD, TANH>(pass, a, nc, ec, grid, s);
    NCN_PICK(false, false, true) NCN_PICK(false, true, true) NCN_PICK(false, false, false) NCN_PICK(false, true, false)
    NCN_PICK(true, false, true) NCN_PICK(true, true, true) NCN_PICK(true, false, false) NCN_PICK(true, true, false)
#undef NCN_PICK
    return hipErrorInvalidConfiguration;
}

}  // namespace ncn
