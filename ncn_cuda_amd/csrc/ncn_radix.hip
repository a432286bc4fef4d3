// Planning and launching of multi-stage passes over levels of the radix-n digit grouping
// (ncn_triton/group_tensors.py:8-18); the kernels are those of ncn_radix_kernels.h, built in ncn_radix_build.hip, and in
// launches with few workgroups the RADIX builds of ncn_fused_kernels.h (ncn_radix_lds.hip).
#include <algorithm>
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

// Whether a pass runs on the kernels that keep rows in LDS, in `lds` workgroups of `rows` rows each, or in `registers` workgroups on
// those that hold `cap` rows in registers.  A lane of the latter holds 16 elements and more, and a workgroup takes the same time
// however few of its rows exist; the former spread the rows there are over 8 waves, 8 elements to a lane, which is the shorter chain as
// long as the workgroups start at once: two to a CU (one on heads of 64 and more) against three.
//   Forward and inverse of tanh, us in LDS : in registers by workgroups (lds, registers).  Groups of two, heads of 8, 6 levels, 64 of
// 1024 rows: (256, 16) 7.5 : 15.9, (512, 32) 9.0 : 15.9, (1024, 64) 16.3 : 16.3; 576 rows: (256, 144) 13.6 : 17.8, (512, 288) 20.5 : 27.3;
// heads of 32, 5 levels, 96 of 256 rows: (512, 192) 14.3 : 13.2, (576, 216) 19.5 : 13.5; 8 levels, all rows: (256, 256) 22.6 : 18.5; heads
// of 64, 5 levels, 32 of 128 rows: (256, 64) 10.0 : 12.5, (512, 128) 18.0 : 13.2.  So a pair on a CU takes 1.2 times as long as one workgroup,
// more the fuller it is of rows, a workgroup longer with more rows, and one more in registers 0.6 of the first; their ratio is that of
// the chains.
//   The other activations spend more instructions on an element, and either kind takes whole rounds of what starts at once: relu,
// groups of two, heads of 8, 5 levels, 32 rows: (512, 16) 14 : 36, (1024, 32) 25 : 36, (2048, 64) 48 : 36; heads of 32, 8 levels, all 256
// rows: (512, 512) 49 : 60, (1024, 1024) 88 : 115; groups of four, heads of 8, 256 of 1024 rows: (512, 128) 22 : 30, (1024, 256) 40 : 33.
//   Over 8684 passes of 16 to 16384 workgroups the choice takes 0.1 % longer than the better of the two, at
// most 15 %.
//   Backward, tanh, groups of two, heads of 8, 8 rows, 3 levels (256, 4) 11.2 : 12.8, (1024, 16) 21.1 : 13.0; heads of 32: 10.8 : 11.3,
// 128 rows, 7 levels (256, 256) 23.3 : 19.3; groups of four, heads of 32, 64 rows, 3 levels (256, 128) 15.3 : 17.4, (512, 256)
// 19.3 : 18.2.  Others, heads of 32, all 128 rows, registers over LDS: 64 workgroups 1.28, 256 1.24, 512 0.77; heads of 64 0.87 at 64.
bool rows_in_lds(int nc, int ec, bool backward, bool tanh, uint32_t rows, uint32_t cap, int64_t lds, int64_t registers) {
    const bool half = 2 * rows <= cap, wide = ec > 32;
    if (backward) return lds <= 256 && (tanh ? half && (ec <= 16 || (ec <= 32 && nc == 4)) : !wide);
    if (lds > 4096) return false;
    auto rounds = [](int64_t workgroups, int64_t at_once) { return (double)((workgroups + at_once - 1) / at_once); };
    if (tanh && wide) return lds <= 256 && half;
    if (tanh) {
        if (5 * rows > 4 * cap) return false;
        const double full = (double)rows / cap, per_cu = rounds(lds, 256), pairs = std::floor(per_cu / 2);
        const double in_lds = (pairs * (1.2 + 1.1 * full) + (per_cu - 2 * pairs)) * (1 + 1.2 * full * full);
        return in_lds < (ec <= 16 ? 2.4 : 2.05) * (1 + 0.6 * (rounds(registers, 256) - 1));
    }
    // time of a round in LDS over one in registers
    const double round = wide ? 0.7 : nc == 4 && ec == 8 ? (half ? 0.75 : 1.1) : half ? 0.42 : 0.66;
    return round * rounds(lds, wide ? 256 : 512) < rounds(registers, 768);
}

RadixLoads radix_loads(const ncn_shape* sh, const RadixPass& p, bool backward, bool tanh) {
    const uint32_t cap = capacity_rows((int)(sh->E / sh->n_head), backward);
    const int64_t whole = sh->batch * (int64_t)p.loads, per = cap / p.span;
    const int64_t across = (sh->batch * (sh->N / p.span) + per - 1) / per;
    if (rows_in_lds(sh->n_cache, (int)(sh->E / sh->n_head), backward, tanh, p.rows, cap, whole * sh->n_head, std::min(whole, across) * sh->n_head))
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
        for (int k = 0; k < p.count; ++k) a.sub_stride[k] = (int32_t)ipow(nc, k);
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
