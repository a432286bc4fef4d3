// Planning and launching of the multi-stage (LDS-resident) passes; kernels in ncn_fused_kernels.h.
#include <algorithm>
#include <cmath>
#include <vector>

#include "ncn_fused_dispatch.h"

namespace ncn {

namespace {

// the shapes the multi-stage kernels are built for: NCN_FOR_EACH_FUSED_CONFIG (ncn_configs.h), tile shapes as in the
// one-stage table

// One window per workgroup wherever the problem allows: workgroups that start and end on their own fall out of step
// with their neighbours on the CU, so that the loads and stores of one run under the stages of the other; a workgroup
// that loops over several windows keeps the phase it started in (measured on the 13-stage configuration: grids of
// 4096 workgroups, 4.5 windows each, 5.35 ms per step; one window each 4.94).  The backward is further bounded by its
// dW partial rows (one per n_head workgroups and stage), see fused_backward_grid.
constexpr int kFusedMaxGridBwd = 1 << 16;
// Windows of a forward launch: a launch holds less than 2^32 work-items.  More windows are given to several launches, by batch entries
// (each of 4 groups of four rows, heads of 8: from 1.07e9 elements on).
constexpr int64_t kFusedMaxGridFwd = ((int64_t(1) << 32) - 1) / (64 * kFusedWavesFwd);
static_assert(kQuadWavesFwd <= kFusedWavesFwd, "threads of a forward workgroup");

size_t fused_lds_bytes(int nc, int ec, bool backward, uint32_t window, int n_stages) {
    const TileShape t = fast_tile(nc, ec);
    const int lr = nc / t.r;
    // groups of two rows keep their slot-0 rows in registers (ncn_fused_pair_kernels.h): one row per group in LDS
    size_t bytes = nc == 2 ? pair_state_bytes(backward) / 2   // the arrays of the largest window, whatever this one's size
                           : (size_t)(backward ? 4 : 2) * window * nc * ec * sizeof(float);
    bytes += (size_t)kFusedMaxStages * 2 * ec * sizeof(float);  // the pass's weights
    const int nw = backward ? (nc == 2 ? kPairWavesBwd : kFusedWavesBwd) : kFusedWavesFwd;
    if (lr > 1) bytes += (size_t)nw * t.f * 64 * sizeof(float);
    if (backward) bytes += (size_t)nw * n_stages * 2 * ec * sizeof(float);
    return bytes;
}

uint32_t stage_stride_of(int stage, uint32_t groups) {
    if (stage == 0) return 0;
    uint64_t r = 1 % groups, b = 2 % groups;
    for (uint32_t e = (uint32_t)stage - 1; e; e >>= 1) {   // 2^(stage-1) mod groups by square and multiply
        if (e & 1) r = r * b % groups;
        b = b * b % groups;
    }
    return (uint32_t)r;
}

uint32_t floor_pow2(uint32_t v) {
    uint32_t p = 1;
    while (p * 2 <= v) p *= 2;
    return p;
}

}  // namespace

bool fused_supported(const ncn_shape* sh, int activation) {
    (void)activation;  // every activation has a build (tanh its own, without the branch on the code)
    const int64_t ec = sh->E / sh->n_head;
    const uint32_t groups = (uint32_t)(sh->N / sh->n_cache);
    // classes are residues modulo a power of two that divides the number of groups: an odd number of groups has none
    if (groups < 2 || (groups & 1u)) return false;
#define NCN_MATCH(NC, EC) \
    if (sh->n_cache == NC && ec == EC) return true;
    NCN_FOR_EACH_FUSED_CONFIG(NCN_MATCH)
#undef NCN_MATCH
    return false;
}

namespace {

// What a halo pass is planned with.  kBothSides: (n_cache - 1) sum(strides) groups on either side of the owned ones, what windows
// of plain sub-blocks would need.  The cuts that ncn_plan_passes reports, and the workspaces that follow from them, are made
// that way; the launch loads the groups that sheared windows need beside the owned ones, which are never more.
// kSheared: those alone, so that halo passes hold more stages.
enum class Halo { kBothSides, kSheared };

// Prices and shapes the passes over stages [a, b) of a range (counted from `first`).  Window capacity in sub-blocks is a
// power of two.
class PassPlanner {
  public:
    PassPlanner(const ncn_shape* sh, int first, int count, bool backward, Halo halo)
        : nc_(sh->n_cache), ec_((int)(sh->E / sh->n_head)), heads_(sh->n_head), groups_((uint32_t)(sh->N / sh->n_cache)), backward_(backward),
          halo_(halo), s_(count) {
        const size_t state = nc_ == 2 ? pair_state_bytes(backward) : fused_state_bytes(backward);
        cap_rows_ = (uint32_t)(state / ((backward ? 4 : 2) * ec_ * sizeof(float)));
        cap_ = floor_pow2(cap_rows_ / nc_);
        if (cap_ > groups_) cap_ = floor_pow2(groups_);
        groups_pow2_ = groups_ & (~groups_ + 1u);   // the power of two in the number of groups
        for (int k = 0; k < count; ++k) s_[k] = stage_stride_of(first + k, groups_);

        // backward keeps a dW slot per wave and stage in LDS: 7 stages leave room for two workgroups per CU at heads of up
        // to 32 features; the two-row kernels at heads of 64 take as many stages as still let two workgroups share a CU
        // (3), at heads of 128 not even two stages would and a CU runs one workgroup of up to 7 stages
        max_stages_ = backward ? kFusedMaxStages - 1 : kFusedMaxStages;
        if (backward && nc_ == 2) {
            const size_t budget = 80 * 1024, fixed = pair_state_bytes(true) / 2 + (size_t)kFusedMaxStages * 2 * ec_ * sizeof(float);
            const size_t per_stage = (size_t)kPairWavesBwd * 2 * ec_ * sizeof(float);
            const int fit = fixed < budget ? (int)((budget - fixed) / per_stage) : 0;
            if (fit >= 2 && fit < max_stages_) max_stages_ = fit;
        }
    }
    int max_stages() const { return max_stages_; }
    // a one-stage launch is bound by its traffic: every array once.  writes_state (backward): the launch hands the
    // reconstructed inputs on.
    double single(bool writes_state) const { return backward_ ? (writes_state ? 8.0 : 6.0) : 4.0; }
    // stages [a, b) as one pass; returns its cost, or < 0 if impossible
    double make(int a, int b, bool writes_state, FusedPass& p) const {
        if (cap_ < 4 || b - a > max_stages_ || b - a < 2) return -1.0;
        // S0: the largest power of two that divides every non-zero stride of the pass and the number of groups (with a
        // power of two of groups the strides are powers of two and this is the smallest of them; with 3 * 2^k groups
        // and the like the strides past 2^k wrap to odd multiples of 2^k)
        uint32_t s0 = 0;
        for (int k = a; k < b; ++k)
            if (s_[k]) {
                const uint32_t low = s_[k] & (~s_[k] + 1u);
                if (!s0 || low < s0) s0 = low;
            }
        if (s0 > groups_pow2_) s0 = groups_pow2_;
        if (!s0) {  // only contiguous-block stages: any class structure works, take full windows
            s0 = groups_pow2_;
            while (s0 > 1 && groups_ / s0 < cap_) s0 /= 2;
        }
        p.first = a;
        p.count = b - a;
        p.single = 0;
        p.class_stride = s0;
        p.ring = groups_ / s0;
        uint32_t sum = 0;
        for (int k = a; k < b; ++k) {
            if (s_[k] % s0) return -1.0;
            p.sub_stride[k - a] = s_[k] / s0;
            sum += s_[k] / s0;
        }
        if (p.ring <= cap_rows_ / nc_) {  // closed: whole rings of adjacent classes, a power of two of them per window
            uint32_t rings = floor_pow2((cap_rows_ / nc_) / p.ring);
            if (rings > s0) rings = s0;
            p.closed = 1;
            p.window = rings * p.ring;
            p.halo = 0;
            p.own = p.window;
            p.tiles_per_ring = 1;
            p.class_groups = s0 / rings;
            if (!fits_launch(p)) return -1.0;
            return priced(writes_state, 1.0, 1.0, b - a, true);
        }
        p.closed = 0;
        p.class_groups = s0;
        // Stage k + 1 of the pass needs slot o of the groups o * step further on than stage k left them (steps around the
        // ring the shorter way): what the window holds beside the owned groups in the stage that runs first, and what all
        // stages do in beside them (`extra`, summed over the stages).
        const uint32_t reach = (uint32_t)nc_ - 1;
        uint64_t extra = 0;
        p.before = p.after = 0;
        p.shear[0] = 0;
        for (int k = 1; k < b - a; ++k) {
            const uint32_t up = (p.sub_stride[k] + p.ring - p.sub_stride[k - 1] % p.ring) % p.ring, down = p.ring - up;
            const bool forth = up <= down;
            p.shear[k] = p.shear[k - 1] + (forth ? (int32_t)up : -(int32_t)down);
            (forth ? p.after : p.before) += reach * (forth ? up : down);
            extra += (uint64_t)reach * (forth ? up : down) * k;   // the k stages before the step
            if (p.before + p.after >= cap_) return -1.0;
        }
        if (halo_ == Halo::kBothSides) {
            p.window = cap_;
            p.halo = reach * sum;
            if (2 * p.halo >= cap_) return -1.0;
            p.own = cap_ - 2 * p.halo;
            if (p.own * 4 < cap_ * 3) return -1.0;  // more than a third of the window would be redundant work
            p.tiles_per_ring = (p.ring + p.own - 1) / p.own;
            if (!fits_launch(p)) return -1.0;
            const double redundancy = (double)cap_ / p.own;
            return priced(writes_state, redundancy, redundancy, b - a, false);
        }
        p.halo = p.before + p.after;
        p.tiles_per_ring = (p.ring + cap_ - p.halo - 1) / (cap_ - p.halo);
        p.own = (p.ring + p.tiles_per_ring - 1) / p.tiles_per_ring;   // windows of one size
        p.window = p.own + p.halo;
        if (p.own * 3 < p.window || !fits_launch(p)) return -1.0;
        const double per_ring = (double)p.tiles_per_ring / p.ring;
        return priced(writes_state, 1.0 + per_ring * p.halo, 1.0 + per_ring * (double)extra / (b - a), b - a, false);
    }

  private:
    // the windows of one batch entry in a launch (backward workgroups walk over windows)
    bool fits_launch(const FusedPass& p) const {
        return backward_ || (int64_t)p.class_groups * p.tiles_per_ring * heads_ <= kFusedMaxGridFwd;
    }
    // What a pass costs, in the time one array of the activations' size takes to cross HBM at copy speed.  Traffic: the
    // pass reads 4 (forward 2) arrays of its windows (window / own times the data) and writes as many of its
    // owned rows; a backward pass that hands no reconstructed inputs on writes the two gradients
    // only (callers that want the reconstructed inputs pay two arrays more than priced here).  Issue: every stage costs
    // `per_stage` such units of instruction issue on all groups of its windows (measured per kernel family on
    // x[128, 8192, 128]: a two-row backward stage 0.143 ms against 0.102 ms per array, a two-row forward stage 0.078 ms;
    // the four-row kernels in proportion to their instruction counts).  The two overlap, better the more they differ:
    // the cube root of the sum of cubes follows the measured pass times to 5 % (a closed backward pass, whose windows
    // are the most scattered in memory, takes 1.1 times that).
    // loaded, computed: windows' share of the groups loaded, and done in a stage on average, over the owned ones
    double priced(bool writes_state, double loaded, double computed, int stages, bool closed) const {
        const double arrays_in = backward_ ? 4.0 : 2.0, arrays_out = backward_ && writes_state ? 4.0 : 2.0;
        const double per_stage = nc_ == 2 ? (backward_ ? 1.4 : 0.76) : (backward_ ? 3.6 : 2.0);
        const double traffic = arrays_in * loaded + arrays_out;
        const double issue = per_stage * stages * computed;
        return std::cbrt(traffic * traffic * traffic + issue * issue * issue) * (closed && backward_ ? 1.1 : 1.0);
    }

    int nc_, ec_, heads_;
    uint32_t groups_, cap_rows_, cap_, groups_pow2_;
    bool backward_;
    Halo halo_;
    int max_stages_;
    std::vector<uint32_t> s_;
};

// One direction of a range whose planning tables are asked for again and again: the cheapest cut of [from, b) into
// passes for every b, the pass at `from` handing no reconstructed inputs on.
struct CheapestCut {
    int from;
    std::vector<double> cost;   // [b - from]
    std::vector<int> last;      // where the last pass of [from, b) begins
    template <class PassCost>
    CheapestCut(int from_, int to, int max_stages, PassCost pass_cost)
        : from(from_), cost(to - from_ + 1, 1e30), last(to - from_ + 1, -1) {
        cost[0] = 0.0;
        for (int b = from + 1; b <= to; ++b)
            for (int a = b - 1; a >= from && (b - a == 1 || b - a <= max_stages); --a) {
                const double c = pass_cost(a, b, a != from);
                if (c >= 0.0 && cost[a - from] + c < cost[b - from] - 1e-9) {
                    cost[b - from] = cost[a - from] + c;
                    last[b - from] = a;
                }
            }
    }
};

FusedPass pass_of(const PassPlanner& planner, int a, int b) {
    FusedPass p{};
    if (b - a > 1) {
        planner.make(a, b, true, p);
    } else {
        p.first = a;
        p.count = 1;
        p.single = 1;
    }
    return p;
}

std::vector<FusedPass> passes_of(const PassPlanner& planner, const CheapestCut& cut, int to) {
    std::vector<FusedPass> passes;
    for (int b = to; b > cut.from; b = cut.last[b - cut.from])
        passes.insert(passes.begin(), pass_of(planner, cut.last[b - cut.from], b));
    return passes;
}

}  // namespace

// Cuts stages [first, first + count) into passes, ascending.
std::vector<FusedPass> plan_fused(const ncn_shape* sh, int first, int count, bool backward, bool sheared) {
    const PassPlanner planner(sh, first, count, backward, sheared ? Halo::kSheared : Halo::kBothSides);
    FusedPass p{};
    const CheapestCut cut(0, count, planner.max_stages(), [&](int a, int b, bool writes_state) {
        return b - a == 1 ? planner.single(writes_state) : planner.make(a, b, writes_state, p);
    });
    return passes_of(planner, cut, count);
}

// Where a stack that is trained keeps its activations.  The forward hands the values between two passes through memory
// anyway: kept, they spare the backward the two arrays that a pass which starts there would otherwise write (and
// the next one read back all the same).  Where both directions' passes begin and end is chosen together, by the prices
// above.  kKeep is what a kept range must gain to be worth its memory.
// With sheared windows, a training step against the cuts of two-sided halos: x[128, 8192, 128] float32, groups of 2, 13 stages, two
// passes in either direction, {0-5} {6-12}, where the forward ran {0-4} {5-12} and the backward {0-2} {3-5} {6-12}: 4255 -> 3672 us;
// x[64, 2048, 128] bfloat16, groups of 4, 6 stages, {0-2} {3-5} in place of {0,1} {2} {3} {4,5} and {0,1} {2} {3} {4} {5}:
// 769 -> 634; x[32, 1024, 128] float32, groups of 4, 5 stages, {0-2} {3,4}: 179 to 189 -> 167.
std::vector<StackRange> plan_stack(const ncn_shape* sh, int first, int count, bool multi_stage, int max_range, int max_saves) {
    constexpr double kKeep = 0.25;
    const PassPlanner fwd(sh, first, count, false, Halo::kSheared), bwd(sh, first, count, true, Halo::kSheared);
    const int F = multi_stage ? fwd.max_stages() : 1, B = multi_stage ? bwd.max_stages() : 1;
    // prices of every pass, made once: [a][length], backward with and without handing the state on
    std::vector<double> fc((size_t)count * (kFusedMaxStages + 1), -1.0), bc(2 * fc.size(), -1.0);
    auto at = [](int a, int len) { return (size_t)a * (kFusedMaxStages + 1) + len; };
    for (int a = 0; a < count; ++a)
        for (int len = 1; len <= kFusedMaxStages && a + len <= count; ++len) {
            FusedPass p{};
            if (len <= F) fc[at(a, len)] = len == 1 ? fwd.single(false) : fwd.make(a, a + len, false, p);
            if (len <= B)
                for (int w = 0; w < 2; ++w)
                    bc[2 * at(a, len) + w] = len == 1 ? bwd.single(w != 0) : bwd.make(a, a + len, w != 0, p);
        }
    std::vector<CheapestCut> fcut, bcut;
    for (int a = 0; a < count; ++a) {
        const int to = a + max_range < count ? a + max_range : count;
        fcut.emplace_back(a, to, F, [&](int u, int v, bool) { return fc[at(u, v - u)]; });
        bcut.emplace_back(a, to, B, [&](int u, int v, bool w) { return bc[2 * at(u, v - u) + (w ? 1 : 0)]; });
    }
    // best[k][b]: [0, b) in k ranges
    std::vector<std::vector<double>> best(max_saves + 1, std::vector<double>(count + 1, 1e30));
    std::vector<std::vector<int>> from(max_saves + 1, std::vector<int>(count + 1, -1));
    best[0][0] = 0.0;
    for (int k = 1; k <= max_saves; ++k)
        for (int b = k; b <= count; ++b)
            for (int a = b - 1; a >= 0 && b - a <= max_range; --a) {
                const double c = best[k - 1][a] + fcut[a].cost[b - a] + bcut[a].cost[b - a] + kKeep;
                if (c < best[k][b] - 1e-9) {
                    best[k][b] = c;
                    from[k][b] = a;
                }
            }
    int k = 0;
    for (int j = 1; j <= max_saves; ++j)
        if (best[j][count] < 1e29 && (k == 0 || best[j][count] < best[k][count])) k = j;
    std::vector<StackRange> ranges(k);
    for (int b = count; k > 0; --k) {
        const int a = from[k][b];
        ranges[k - 1] = StackRange{passes_of(fwd, fcut[a], b), passes_of(bwd, bcut[a], b)};
        b = a;
    }
    return ranges;
}

int64_t fused_items(const ncn_shape* sh, const FusedPass& p) {
    return sh->batch * (int64_t)p.class_groups * p.tiles_per_ring * sh->n_head;
}

int fused_backward_grid(const ncn_shape* sh, const FusedPass& p, int row_cap) {
    const int64_t cap = std::min<int64_t>(kFusedMaxGridBwd, (int64_t)row_cap / p.count * sh->n_head);
    const int64_t g = std::min(fused_items(sh, p), cap) / sh->n_head * sh->n_head;
    return (int)std::max<int64_t>(g, sh->n_head);
}

namespace {

const void* elements_at(const void* base, int dtype, int64_t at) {
    return base ? static_cast<const char*>(base) + at * (dtype == NCN_F32 ? 4 : 2) : nullptr;
}

}  // namespace

hipError_t launch_fused(Pass pass, FusedArgs& a, const ncn_shape* sh, const FusedPass& p, hipStream_t s, int row_cap,
                        bool headwise) {
    const bool backward = pass == kBackward;
    const int nc = sh->n_cache, ec = (int)(sh->E / sh->n_head);
    a.N = sh->N;
    a.E = sh->E;
    a.n_head = sh->n_head;
    a.n_stages = p.count;
    a.class_stride = p.class_stride;
    a.ring = p.ring;
    a.ring_magic = (p.ring & (p.ring - 1)) == 0 ? 0u : (uint32_t)(((1ull << 32) + p.ring - 1) / p.ring);
    a.own = p.own;
    a.tiles_per_ring = p.tiles_per_ring;
    a.closed = p.closed;
    a.class_groups = p.class_groups;
    if (p.closed) {
        a.window = p.window;
        for (int k = 0; k < p.count; ++k) a.sub_stride[k] = (int32_t)p.sub_stride[k];
    } else {   // the window as the stage that runs first needs it
        const int first = pass == kForward ? 0 : p.count - 1, last = p.count - 1 - first;
        a.window = p.before + p.own + p.after;
        a.halo = pass == kForward ? p.before : p.after;
        a.shift = p.sub_stride[first] % p.ring;
        for (int k = 0; k < p.count; ++k) a.sub_stride[k] = p.shear[k] - p.shear[first];
        a.end_shear = a.sub_stride[last];
    }
    a.scale_dn = (float)std::pow((double)a.tab.m, (double)(nc * p.count));
    a.scale_up = (float)std::pow((double)a.tab.m, -(double)(nc * p.count));
    const size_t lds = fused_lds_bytes(nc, ec, backward, a.window, p.count);
    auto launch = [&](const FusedArgs& args, int grid) {
        if (headwise) return launch_fused_headwise(pass, args, nc, ec, grid, lds, s);
        if (args.ctx_len) return launch_fused_lengths(pass, args, nc, ec, grid, lds, s);
        return launch_fused_shape<false, false, false>(pass, args, nc, ec, grid, lds, s);
    };
    const int64_t items = fused_items(sh, p);
    a.total_items = (uint32_t)items;
    if (backward) return launch(a, fused_backward_grid(sh, p, row_cap));
    // a workgroup for every window
    if (items <= kFusedMaxGridFwd) return launch(a, (int)items);
    const int64_t per_entry = items / sh->batch, entries = kFusedMaxGridFwd / per_entry;   // at least one: fits_launch
    for (int64_t b = 0; b < sh->batch; b += entries) {
        const int64_t at = b * sh->N * sh->E, n = std::min(entries, sh->batch - b) * per_entry;
        FusedArgs part = a;
        part.in0 = elements_at(a.in0, a.in_dtype, at);
        part.in1 = elements_at(a.in1, a.in_dtype, at);
        part.out0 = const_cast<void*>(elements_at(a.out0, a.out_dtype, at));
        part.out1 = const_cast<void*>(elements_at(a.out1, a.out_dtype, at));
        part.aux0 = a.aux0 ? a.aux0 + at : nullptr;
        part.aux1 = a.aux1 ? a.aux1 + at : nullptr;
        part.ctx_len = a.ctx_len ? a.ctx_len + b : nullptr;
        part.total_items = (uint32_t)n;
        const hipError_t err = launch(part, (int)n);
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}

}  // namespace ncn
