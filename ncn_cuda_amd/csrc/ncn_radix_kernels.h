// Several levels of the radix-n digit grouping (ncn_triton/group_tensors.py:8-18) per pass, on rows that stay in registers;
// groups of 2 and 4 rows.
//
// Which rows.  Level l groups the n_cache positions that differ only in base-n_cache digit l.  A run of levels a .. a+k-1
// only ever mixes the positions lower + n^a d + n^(a+k) upper, d = 0 .. n^k - 1, of one (lower, upper): a closed window of n^k
// rows, no halo, any pass may run in place.  A workgroup holds rows / n^k such windows; row lr of a workgroup is window
// lr / n^k, digit string d = lr mod n^k.  (Every size but the number of windows is a power of two.)
//
// Where they are.  A level on a digit is a butterfly over that digit's bits of lr, and the kernels go through the levels as an
// FFT does: the bits of a row number ("slot") are spread over the registers of a lane (RB bits), the row lanes of a wave (LB)
// and the waves of a workgroup (WB), and a level runs where its bits are register bits: all rows of a group in one lane, the
// step code of ncn_stage_kernels.h without any exchange between rows.  Then register bits and lane bits change places:
// v_permlane32_swap and v_permlane16_swap exchange the upper two lane bits with a register bit in one instruction per two
// registers, DPP moves the lower ones.  What lies across waves comes in by an exchange of all rows through LDS after the
// RB + LB bits before it (heads of 32, groups of two: six levels forward, five backward; heads of 128, groups of four, backward:
// one).  (The RADIX builds of ncn_fused_kernels.h keep the rows in LDS, read and write them all at every level with a
// barrier after it: x[32, 8192, 128], 13 levels of groups of two, 8 + 5 forward and 7 + 6 backward, 231 us a pass forward and 459
// backward; here 213 and 152, 345 and 316.  They run where there are few workgroups: rows_in_lds() in ncn_radix.hip.)
//
// What bounds it: of the 345 us of the backward pass over 7 levels its loads, stores and exchanges alone take 174, its
// instructions at the rates they issue at some 210, and with four workgroups per CU, whose registers are full, the two overlap
// only so far.  The forward holds twice the elements at three waves per SIMD (150 registers); with half of them at six waves a
// training pass took 914 us instead of 900, at four waves with 24 spilled registers 940.
//
// Bits are numbered in the order the levels run in: logical bit q is the q-th to be a register bit, so digit count-1 comes
// first where levels are undone (backward, inverse).  RadixMap says where each logical bit is; all of it is known at compile
// time but the number of levels of the pass: bits past them number windows and are carried along.
#pragma once
#include "ncn_fused_kernels.h"
#include "ncn_fused_pair_kernels.h"

namespace ncn {

template <int NC, int EC, bool BACKWARD>
struct RadixShape {
    static constexpr int DB = NC == 2 ? 1 : 2;                    // bits of a digit
    // 8 features per lane (row sums cross half the lanes of 4, and what is paid per row is spread over twice the elements);
    // forward 4 rows of them (32 elements of two arrays), backward 2 (16 of four), or 4 rows of 4 where a group has 4.  Heads
    // of 8 features have 4 to a lane and twice the rows: lane bits inside a quad cost four instructions where the others cost
    // one or two (x[64, 4096, 32], 12 levels, groups of two: 404 us a training pass, 419 with 8)
    static constexpr int F = EC == 8 || (BACKWARD && NC == 4) ? 4 : 8;
    static constexpr int RB = BACKWARD ? (NC == 2 && EC > 8 ? 1 : 2) : (NC == 2 && EC == 8 ? 3 : 2);   // register bits
    static constexpr int R = 1 << RB;                             // rows per lane
    static constexpr int H = F / 4;                               // 16-byte chunks per lane and row: fl, fl + LF
    static constexpr int LF = EC / F, LG_LF = LF == 1 ? 0 : LF == 2 ? 1 : LF == 4 ? 2 : LF == 8 ? 3 : LF == 16 ? 4 : 5;
    static constexpr int LB = 6 - LG_LF;                          // row bits of a lane
    static constexpr int WB = !BACKWARD && NC == 4 && EC == 8 ? 3 : 2, NW = 1 << WB;   // waves of a workgroup: 64 KB of rows in registers
    static constexpr int T = RB + LB + WB;                        // bits of a slot
    static constexpr int TU = T / DB * DB;                        // .. that whole digits can use
    static_assert(LF * F == EC && (1 << LG_LF) == LF && LB >= 0, "a row fits the lanes of a wave");
};

// where[q]: position of logical bit q -- register bits, then row bits of the lane, then bits of the wave's number
struct RadixMap {
    int where[12];
};
// positions at the start of the phase that takes up logical bit p0, after its first `chunks` exchanges of register and lane bits
template <class S>
constexpr RadixMap radix_map(int p0, int chunks) {
    RadixMap m{};
    for (int k = 0; k < S::T; ++k) m.where[(p0 + k) % S::T] = k;
    for (int c = 0; c < chunks; ++c)
        for (int i = 0; i < S::RB; ++i) {
            const int lane_pos = S::RB + c * S::RB + i;
            if (lane_pos >= S::RB + S::LB) break;
            for (int q = 0; q < S::T; ++q) m.where[q] = m.where[q] == i ? lane_pos : m.where[q] == lane_pos ? i : m.where[q];
        }
    return m;
}
// exchanges of the phase that begins at p0, each of RB lane bits (groups of 4 rows need both bits of a digit), as long as there
// are bits left to take up
template <class S>
constexpr int radix_chunks(int p0) {
    const int all = S::DB == 1 ? (S::LB + S::RB - 1) / S::RB : S::LB / S::RB;
    const int need = S::TU - p0 > S::RB ? (S::TU - p0 - S::RB + S::RB - 1) / S::RB : 0;
    return need < all ? need : all;
}
// logical bits done after the phase that began at p0
template <class S>
constexpr int radix_done(int p0) {
    const int p = p0 + S::RB + (S::DB == 1 ? S::LB : S::LB / S::RB * S::RB);
    return p < S::TU ? p : S::TU;
}
// slot bits that register r stands for
template <class S>
constexpr uint32_t radix_reg_slot(const RadixMap& m, int r) {
    uint32_t s = 0;
    for (int q = 0; q < S::T; ++q)
        if (m.where[q] < S::RB && (r >> m.where[q]) & 1) s |= 1u << q;
    return s;
}
// .. and those of the lane and the wave
template <class S, int P0, int CHUNKS>
__device__ __forceinline__ uint32_t radix_lane_slot(int lane, int wave) {
    constexpr RadixMap m = radix_map<S>(P0, CHUNKS);
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < S::T; ++q) {
        const int w = m.where[q];
        if (w >= S::RB + S::LB) s |= (((uint32_t)wave >> (w - S::RB - S::LB)) & 1u) << q;
        else if (w >= S::RB) s |= (((uint32_t)lane >> (S::LG_LF + w - S::RB)) & 1u) << q;
    }
    return s;
}

// Row number of a slot (linear in its bits).  DESC: the first logical digit is the highest of the pass.
template <int DB, bool DESC>
__device__ __forceinline__ uint32_t radix_row(uint32_t slot, int count) {
    if (!DESC) return slot;
    const int bits = count * DB;
    const uint32_t mask = (1u << bits) - 1u;
    uint32_t rev = __brev(slot & mask) >> (32 - bits);
    if (DB == 2) rev = ((rev & 0xaaaaaaaau) >> 1) | ((rev & 0x55555555u) << 1);   // digits reversed, not their bits
    return (slot & ~mask) | rev;
}

// a, b are two registers that differ in a register bit: afterwards that bit and lane bit BIT have changed places, i.e. lanes
// whose bit is 0 hold a of both lanes, lanes whose bit is 1 hold b of both
template <int BIT>
__device__ __forceinline__ void radix_swap(float& a, float& b, int lane) {
    if constexpr (BIT == 5) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    } else if constexpr (BIT == 4) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    } else {
        const int x = __float_as_int(a), y = __float_as_int(b);
        int na, nb;
        if constexpr (BIT == 3) {   // row_ror:8 reads lane ^ 8; banks 2, 3 have the bit set
            na = __builtin_amdgcn_update_dpp(x, y, 0x128, 0xF, 0xC, false);
            nb = __builtin_amdgcn_update_dpp(y, x, 0x128, 0xF, 0x3, false);
        } else if constexpr (BIT == 2) {   // row_shr:4 reads lane - 4 (banks 1, 3), row_shl:4 lane + 4 (banks 0, 2)
            na = __builtin_amdgcn_update_dpp(x, y, 0x114, 0xF, 0xA, false);
            nb = __builtin_amdgcn_update_dpp(y, x, 0x104, 0xF, 0x5, false);
        } else {   // inside a quad: lane ^ 2 or lane ^ 1, no mask picks the lanes
            constexpr int perm = BIT == 1 ? 0x4E : 0xB1;
            const int px = __builtin_amdgcn_mov_dpp(x, perm, 0xF, 0xF, true), py = __builtin_amdgcn_mov_dpp(y, perm, 0xF, 0xF, true);
            const bool set = (lane >> BIT) & 1;
            na = set ? py : x;
            nb = set ? y : px;
        }
        a = __int_as_float(na);
        b = __int_as_float(nb);
    }
}

// chunk C of a phase: register bit i changes places with row bit C * RB + i of the lane
template <class S, int C, int I = 0>
__device__ __forceinline__ void radix_exchange(float (&v)[S::R][S::F], int lane) {
    if constexpr (I < S::RB && C * S::RB + I < S::LB) {
#pragma unroll
        for (int r = 0; r < S::R; ++r) {
            if ((r >> I) & 1) continue;
#pragma unroll
            for (int f = 0; f < S::F; ++f) radix_swap<S::LG_LF + C * S::RB + I>(v[r][f], v[r | (1 << I)][f], lane);
        }
        radix_exchange<S, C, I + 1>(v, lane);
    }
}

// Through LDS: the array as it lies after a phase to where the next one wants it.  A row's chunks are rotated by the bits of
// its slot, or the rows of a wave, a multiple of 32 banks apart, would all start in the same bank.
template <int EC>
__device__ __forceinline__ uint32_t radix_lds_chunk(uint32_t slot, uint32_t chunk) {
    constexpr uint32_t CPR = EC / 4;
    return slot * CPR + (chunk ^ ((slot ^ (slot >> 2) ^ (slot >> 4)) & (CPR - 1u)));
}
template <class S, int EC, int P0, int P1>
__device__ __forceinline__ void radix_remap(float (&v)[S::R][S::F], float4* exch, int lane, int wave, int fl) {
    constexpr RadixMap from = radix_map<S>(P0, radix_chunks<S>(P0)), to = radix_map<S>(P1, 0);
    const uint32_t s0 = radix_lane_slot<S, P0, radix_chunks<S>(P0)>(lane, wave), s1 = radix_lane_slot<S, P1, 0>(lane, wave);
#pragma unroll
    for (int r = 0; r < S::R; ++r)
#pragma unroll
        for (int h = 0; h < S::H; ++h)
            exch[radix_lds_chunk<EC>(s0 | radix_reg_slot<S>(from, r), fl + h * S::LF)] =
                make_float4(v[r][4 * h], v[r][4 * h + 1], v[r][4 * h + 2], v[r][4 * h + 3]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < S::R; ++r)
#pragma unroll
        for (int h = 0; h < S::H; ++h) {
            const float4 t = exch[radix_lds_chunk<EC>(s1 | radix_reg_slot<S>(to, r), fl + h * S::LF)];
            v[r][4 * h] = t.x; v[r][4 * h + 1] = t.y; v[r][4 * h + 2] = t.z; v[r][4 * h + 3] = t.w;
        }
    __syncthreads();   // the next array takes the same place
}

template <class S>
__device__ __forceinline__ void radix_weights(const float* w, int fl, float (&v)[S::F]) {
#pragma unroll
    for (int h = 0; h < S::H; ++h) {
        const float4 t = *reinterpret_cast<const float4*>(w + (fl + h * S::LF) * 4);
        v[4 * h] = t.x; v[4 * h + 1] = t.y; v[4 * h + 2] = t.z; v[4 * h + 3] = t.w;
    }
}

// The windows of a workgroup: of one batch entry where a divisor of their number fills it, else (class_groups 0) counted through
// all batch entries, so that short sequences fill workgroups too.  x[4096, 32, 128], 5 levels of groups of two, forward, us: 32 rows
// of the 256 that a workgroup holds 426, all of them 82; x[512, 640, 128], 7 levels (windows of 128 rows, five to an entry) 385
// with one to a workgroup, 231 with two.
struct RadixItem {
    int head;
    uint32_t window0, rows;   // first window, in its batch entry; rows that exist
    int64_t base;             // element offset of (batch entry, row 0, head slice)
};
template <int NC, int EC>
__device__ __forceinline__ RadixItem radix_item(const FusedArgs& A, uint32_t item) {
    RadixItem it;
    it.head = item % A.n_head;
    const uint32_t load = item / A.n_head, per = (A.window * NC) >> log2u(A.ring);
    uint32_t b;
    it.rows = A.window * NC;
    if (A.class_groups) {
        b = load / A.class_groups;
        it.window0 = (load - b * A.class_groups) * per;
    } else {
        const uint32_t w = load * per;
        b = w / A.entry_windows;
        it.window0 = w - b * A.entry_windows;
        it.rows = min(per, A.all_windows - w) << log2u(A.ring);
    }
    it.base = (int64_t)b * A.N * A.E + (int64_t)it.head * EC;
    return it;
}
// element offset (without the feature) of row lr of a workgroup
__device__ __forceinline__ int64_t radix_row_offset(const FusedArgs& A, const RadixItem& it, uint32_t lr) {
    const uint32_t lg_span = log2u(A.ring), lg_s0 = log2u(A.class_stride);
    const uint32_t d = lr & (A.ring - 1u);
    uint32_t u = it.window0 + (lr >> lg_span);
    int64_t base = it.base;
    if (A.class_groups == 0u) {   // u may lie in a later entry: the next, or, where a workgroup holds several, the u / entry_windows-th
        const uint32_t k = A.entry_magic ? __umulhi(2u * u, A.entry_magic) : u >= A.entry_windows ? 1u : 0u;
        u -= k * A.entry_windows;
        base += (int64_t)k * (A.N * A.E);
    }
    const int64_t pos = (int64_t)(u & (A.class_stride - 1u)) + ((int64_t)d << lg_s0) + ((int64_t)(u >> lg_s0) << (lg_s0 + lg_span));
    return base + pos * A.E;
}

// Offsets of this lane's rows as they lie after `CHUNKS` exchanges of phase P0; a row that does not exist (the windows of the
// workgroup do not fill it) gets row 0's and its bit of the result is 0.
template <class S, int NC, int P0, int CHUNKS, bool DESC>
__device__ __forceinline__ uint32_t radix_offsets(const FusedArgs& A, const RadixItem& it, int lane, int wave, int fl,
                                                  int64_t (&off)[S::R]) {
    constexpr RadixMap m = radix_map<S>(P0, CHUNKS);
    const uint32_t base = radix_row<S::DB, DESC>(radix_lane_slot<S, P0, CHUNKS>(lane, wave), A.n_stages);
    uint32_t exists = 0;
#pragma unroll
    for (int r = 0; r < S::R; ++r) {
        const uint32_t lr = base | radix_row<S::DB, DESC>(radix_reg_slot<S>(m, r), A.n_stages);
        const bool ok = lr < it.rows;
        exists |= ok ? 1u << r : 0u;
        off[r] = radix_row_offset(A, it, ok ? lr : 0u) + fl * 4;
    }
    return exists;
}
template <class S>
__device__ __forceinline__ void radix_fetch(const void* src, int dtype, const int64_t (&off)[S::R], uint4 (&raw)[S::R * S::H]) {
    int64_t o[S::R * S::H];
#pragma unroll
    for (int r = 0; r < S::R; ++r)
#pragma unroll
        for (int h = 0; h < S::H; ++h) o[r * S::H + h] = off[r] + h * S::LF * 4;
    fused_fetch_rows<S::R * S::H>(src, dtype, o, raw);
}
template <class S>
__device__ __forceinline__ void radix_commit(const uint4 (&raw)[S::R * S::H], int dtype, float scale, float (&v)[S::R][S::F]) {
#pragma unroll
    for (int r = 0; r < S::R; ++r)
#pragma unroll
        for (int h = 0; h < S::H; ++h) {
            float t[4];
            fused_raw_to_float(raw[r * S::H + h], dtype, t);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[r][4 * h + e] = t[e] * scale;
        }
}
template <class S>
__device__ __forceinline__ void radix_store(void* dst, int dtype, const int64_t (&off)[S::R], uint32_t exists, float scale,
                                            const float (&v)[S::R][S::F]) {
#pragma unroll
    for (int r = 0; r < S::R; ++r)
#pragma unroll
        for (int h = 0; h < S::H; ++h) {
            float t[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = v[r][4 * h + e] * scale;
            store_frag<4>(dst, dtype, off[r] + h * S::LF * 4, (exists >> r) & 1u, t);
        }
}

// ---- forward, and with INVERSE the same levels undone -------------------------------------------------------------
template <int NC, int EC, bool TANH_ONLY, bool INVERSE, bool HEADWISE>
struct RadixForward {
    using S = RadixShape<NC, EC, false>;
    const FusedArgs& A;
    const RadixItem& it;
    const float* w_lds;
    float4* exch;
    int lane, wave, fl;
    float x[S::R][S::F], a[S::R][S::F];

    // one level on the rows that register numbers `r0 + o step` (slot o) name
    template <int STEP>
    __device__ __forceinline__ void group(int r0, const float (&wi)[S::F], const float (&wj)[S::F]) {
        float gx[NC][S::F], ga[NC][S::F];
#pragma unroll
        for (int o = 0; o < NC; ++o)
#pragma unroll
            for (int f = 0; f < S::F; ++f) {
                gx[o][f] = x[r0 + o * STEP][f];
                ga[o][f] = a[r0 + o * STEP][f];
            }
        if constexpr (HEADWISE) {
            if (INVERSE) headwise_inverse_core<NC, EC, NC, S::F, TANH_ONLY, false, true>(gx, ga, wi, wj, A.tab, lane, nullptr);
            else headwise_forward_core<NC, EC, NC, S::F, TANH_ONLY, false, true>(gx, ga, wi, wj, A.tab, lane, nullptr);
        } else {
            if (INVERSE) inverse_core<NC, EC, NC, S::F, TANH_ONLY, false, true>(gx, ga, wi, wj, A.tab, lane, nullptr);
            else forward_core<NC, EC, NC, S::F, TANH_ONLY, false, true>(gx, ga, wi, wj, A.tab, lane, nullptr);
        }
#pragma unroll
        for (int o = 0; o < NC; ++o)
#pragma unroll
            for (int f = 0; f < S::F; ++f) {
                x[r0 + o * STEP][f] = gx[o][f];
                a[r0 + o * STEP][f] = ga[o][f];
            }
    }
    template <int Q, int N, int I = 0>
    __device__ __forceinline__ void levels() {   // logical bits Q .. Q + N - 1, which are the first N register bits
        if constexpr (I < N && Q + I < S::TU) {
            const int d = (Q + I) / S::DB;   // the d-th level to run
            if (d < A.n_stages) {
                const int st = INVERSE ? A.n_stages - 1 - d : d;
                float wi[S::F], wj[S::F];
                radix_weights<S>(w_lds + st * 2 * EC, fl, wi);
                radix_weights<S>(w_lds + st * 2 * EC + EC, fl, wj);
#pragma unroll
                for (int r = 0; r < S::R; ++r)
                    if (((r >> I) & (NC - 1)) == 0) group<(1 << I)>(r, wi, wj);
            }
            levels<Q, N, I + S::DB>();
        }
    }
    template <int P0, int C = 0>
    __device__ __forceinline__ void chunks() {
        if constexpr (C < radix_chunks<S>(P0)) {
            radix_exchange<S, C>(x, lane);
            radix_exchange<S, C>(a, lane);
            constexpr int left = S::LB - C * S::RB;   // the last exchange may bring in fewer bits than there are register bits
            levels<P0 + S::RB + C * S::RB, (left < S::RB ? left : S::RB)>();
            chunks<P0, C + 1>();
        }
    }
    template <int P0 = 0>
    __device__ __forceinline__ void run() {
        levels<P0, S::RB>();
        chunks<P0>();
        constexpr int P1 = radix_done<S>(P0);
        if constexpr (P1 < S::TU) {
            if (A.n_stages * S::DB > P1) {
                radix_remap<S, EC, P0, P1>(x, exch, lane, wave, fl);
                radix_remap<S, EC, P0, P1>(a, exch, lane, wave, fl);
                run<P1>();
                return;
            }
        }
        int64_t off[S::R];
        const uint32_t exists = radix_offsets<S, NC, P0, radix_chunks<S>(P0), INVERSE>(A, it, lane, wave, fl, off);
        const float a_out = INVERSE ? A.tab.inv_b_scale : A.tab.inv_a_scale;
        radix_store<S>(A.out0, A.out_dtype, off, exists, A.tab.inv_kappa, x);
        radix_store<S>(A.out1, A.out_dtype, off, exists, a_out, a);
        if (A.aux0) {
            radix_store<S>(A.aux0, NCN_F32, off, exists, A.tab.inv_kappa, x);
            radix_store<S>(A.aux1, NCN_F32, off, exists, a_out, a);
        }
    }
};

template <int NC, int EC, bool TANH_ONLY, bool INVERSE, bool HEADWISE>
__global__ void __launch_bounds__((64 * RadixShape<NC, EC, false>::NW), TANH_ONLY ? 3 : 1) radix_forward_kernel(const FusedArgs A) {
    using K = RadixForward<NC, EC, TANH_ONLY, INVERSE, HEADWISE>;
    using S = typename K::S;
    extern __shared__ float4 fused_lds4[];
    float* w_lds = reinterpret_cast<float*>(fused_lds4);                  // [kFusedMaxStages][2][EC]
    float4* exch = fused_lds4 + kFusedMaxStages * 2 * EC / 4;             // one array of the workgroup
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fl = lane % S::LF;
    const RadixItem it = radix_item<NC, EC>(A, fused_deal<EC>(A, blockIdx.x));   // the launch has a workgroup for every item
    int64_t off[S::R];
    radix_offsets<S, NC, 0, 0, INVERSE>(A, it, lane, wave, fl, off);
    uint4 rx[S::R * S::H], ra[S::R * S::H];
    radix_fetch<S>(A.in0, A.in_dtype, off, rx);
    radix_fetch<S>(A.in1, A.in_dtype, off, ra);
    fused_load_weights<EC, S::NW>(A, it.head, w_lds);
    K k{A, it, w_lds, exch, lane, wave, fl};
    radix_commit<S>(rx, A.in_dtype, A.tab.kappa, k.x);
    radix_commit<S>(ra, A.in_dtype, INVERSE ? A.tab.b_scale : A.tab.a_scale, k.a);
    __syncthreads();
    k.run();
}

// ---- backward -----------------------------------------------------------------------------------------------------
template <int NC, int EC, bool TANH_ONLY, bool LOOP, bool HEADWISE>
struct RadixBackward {
    using S = RadixShape<NC, EC, true>;
    const FusedArgs& A;
    const RadixItem& it;
    const float* w_lds;
    float* dw_mine;   // [n_stages][2][EC] of this wave
    float4* exch;
    int lane, wave, fl;
    float Y[S::R][S::F], B[S::R][S::F], G[S::R][S::F], P[S::R][S::F];

    template <int STEP>
    __device__ __forceinline__ void group(int r0, int step_base, const float (&wi)[S::F], const float (&wj)[S::F],
                                          float (&dwi)[S::F], float (&dwj)[S::F]) {
        float gy[NC][S::F], gb[NC][S::F], gg[NC][S::F], gp[NC][S::F];
#pragma unroll
        for (int o = 0; o < NC; ++o)
#pragma unroll
            for (int f = 0; f < S::F; ++f) {
                gy[o][f] = Y[r0 + o * STEP][f]; gb[o][f] = B[r0 + o * STEP][f];
                gg[o][f] = G[r0 + o * STEP][f]; gp[o][f] = P[r0 + o * STEP][f];
            }
        if constexpr (HEADWISE)
            headwise_backward_core<NC, EC, NC, S::F, false, TANH_ONLY, false, true, false>(gy, gb, gg, gp, wi, wj, dwi, dwj, 1.0f,
                                                                                        A.tab, step_base, lane, nullptr);
        else
            backward_core<NC, EC, NC, S::F, false, TANH_ONLY, false, true, false>(gy, gb, gg, gp, wi, wj, dwi, dwj, 1.0f, A.tab,
                                                                               step_base, lane, nullptr);
#pragma unroll
        for (int o = 0; o < NC; ++o)
#pragma unroll
            for (int f = 0; f < S::F; ++f) {
                Y[r0 + o * STEP][f] = gy[o][f]; B[r0 + o * STEP][f] = gb[o][f];
                G[r0 + o * STEP][f] = gg[o][f]; P[r0 + o * STEP][f] = gp[o][f];
            }
    }
    // this wave's dW share of level st into its own LDS slot, in a fixed order
    __device__ __forceinline__ void put_dw(int st, float (&dw)[2 * S::F]) {
        float* const slot = dw_mine + st * (2 * EC);
        auto add = [](float* d, float v) { *d = LOOP ? *d + v : v; };   // one item: one value
        if constexpr (S::F == 8) {
            const int first = pair_scatter_sum<S::LF, 16>(dw, lane);
            constexpr int LEFT = pair_scatter_left<S::LF, 16>();
            const int half = first / 8, f0 = first % 8;
            float* d = slot + half * EC + (fl + (f0 / 4) * S::LF) * 4 + (f0 % 4);
            if (S::LF >= 4 || (lane & (S::LF == 2 ? 2 : 3)) == 0) {   // narrow heads: one lane per value writes
#pragma unroll
                for (int i = 0; i < LEFT; ++i) add(d + i, dw[i]);
            }
        } else {
            lane_sum_n<S::LF, 64, true, 2 * S::F>(dw);
            if (lane < S::LF) {
#pragma unroll
                for (int f = 0; f < S::F; ++f) {
                    add(slot + fl * 4 + f, dw[f]);
                    add(slot + EC + fl * 4 + f, dw[S::F + f]);
                }
            }
        }
    }
    template <int Q, int N, int I = 0>
    __device__ __forceinline__ void levels() {   // logical bits Q .. Q + N - 1, which are the first N register bits
        if constexpr (I < N && Q + I < S::TU) {
            const int d = (Q + I) / S::DB;
            if (d < A.n_stages) {
                const int st = A.n_stages - 1 - d;
                float wi[S::F], wj[S::F], dw[2 * S::F];
                radix_weights<S>(w_lds + st * 2 * EC, fl, wi);
                radix_weights<S>(w_lds + st * 2 * EC + EC, fl, wj);
#pragma unroll
                for (int f = 0; f < 2 * S::F; ++f) dw[f] = 0.f;
                float (&dwi)[S::F] = *reinterpret_cast<float (*)[S::F]>(&dw[0]);
                float (&dwj)[S::F] = *reinterpret_cast<float (*)[S::F]>(&dw[S::F]);
#pragma unroll
                for (int r = 0; r < S::R; ++r)
                    if (((r >> I) & (NC - 1)) == 0) group<(1 << I)>(r, d * NC, wi, wj, dwi, dwj);
                put_dw(st, dw);
            }
            levels<Q, N, I + S::DB>();
        }
    }
    template <int P0, int C = 0>
    __device__ __forceinline__ void chunks() {
        if constexpr (C < radix_chunks<S>(P0)) {
            radix_exchange<S, C>(Y, lane);
            radix_exchange<S, C>(B, lane);
            radix_exchange<S, C>(G, lane);
            radix_exchange<S, C>(P, lane);
            constexpr int left = S::LB - C * S::RB;
            levels<P0 + S::RB + C * S::RB, (left < S::RB ? left : S::RB)>();
            chunks<P0, C + 1>();
        }
    }
    template <int P0 = 0>
    __device__ __forceinline__ void run() {
        levels<P0, S::RB>();
        chunks<P0>();
        constexpr int P1 = radix_done<S>(P0);
        if constexpr (P1 < S::TU) {
            if (A.n_stages * S::DB > P1) {
                radix_remap<S, EC, P0, P1>(Y, exch, lane, wave, fl);
                radix_remap<S, EC, P0, P1>(B, exch, lane, wave, fl);
                radix_remap<S, EC, P0, P1>(G, exch, lane, wave, fl);
                radix_remap<S, EC, P0, P1>(P, exch, lane, wave, fl);
                run<P1>();
                return;
            }
        }
        // true values: g = G m^T, h = P m^T - (1-m) g, x = xs / kappa, xa = bh / b_scale
        int64_t off[S::R];
        const uint32_t exists = radix_offsets<S, NC, P0, radix_chunks<S>(P0), true>(A, it, lane, wave, fl, off);
#pragma unroll
        for (int r = 0; r < S::R; ++r)
#pragma unroll
            for (int f = 0; f < S::F; ++f) {
                G[r][f] *= A.scale_dn;
                P[r][f] = fmaf(P[r][f], A.scale_dn, -A.tab.om * G[r][f]);
            }
        radix_store<S>(A.out0, A.out_dtype, off, exists, 1.0f, G);
        radix_store<S>(A.out1, A.out_dtype, off, exists, 1.0f, P);
        if (A.aux0) {
            radix_store<S>(A.aux0, NCN_F32, off, exists, A.tab.inv_kappa, Y);
            radix_store<S>(A.aux1, NCN_F32, off, exists, A.tab.inv_b_scale, B);
        }
    }
};

// LOOP: for calls with more items than the dW scratch has partial rows; at four waves per SIMD the loop spills 32 registers (x[128, 8192,
// 128], 13 levels: 3688 us a training pass, 3511 with three)
template <int NC, int EC, bool TANH_ONLY, bool LOOP, bool HEADWISE>
__global__ void __launch_bounds__((64 * RadixShape<NC, EC, true>::NW), TANH_ONLY ? (LOOP ? 3 : 4) : 1) radix_backward_kernel(const FusedArgs A) {
    using K = RadixBackward<NC, EC, TANH_ONLY, LOOP, HEADWISE>;
    using S = typename K::S;
    extern __shared__ float4 fused_lds4[];
    float* w_lds = reinterpret_cast<float*>(fused_lds4);                      // [kFusedMaxStages][2][EC]
    float4* exch = fused_lds4 + kFusedMaxStages * 2 * EC / 4;                 // one array of the workgroup
    float* dw_all = reinterpret_cast<float*>(exch + ((size_t)EC / 4 << S::T));   // [wave][stage][2][EC]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fl = lane % S::LF;
    const int dw_stride = A.n_stages * 2 * EC;
    float* dw_mine = dw_all + wave * dw_stride;
    const uint32_t item0 = LOOP ? blockIdx.x : fused_deal<EC>(A, blockIdx.x);
    const int head = item0 % A.n_head;   // of every item of this workgroup (gridDim.x % n_head == 0)
    if (LOOP)
        for (int k = lane; k < dw_stride; k += 64) dw_mine[k] = 0.f;
    uint32_t item = item0;
    do {
        const RadixItem it = radix_item<NC, EC>(A, item);
        int64_t off[S::R];
        const uint32_t exists = radix_offsets<S, NC, 0, 0, true>(A, it, lane, wave, fl, off);
        uint4 ry[S::R * S::H], rb[S::R * S::H], rg[S::R * S::H], rh[S::R * S::H];
        radix_fetch<S>(A.in0, A.in_dtype, off, ry);
        radix_fetch<S>(A.in1, A.in_dtype, off, rb);
        radix_fetch<S>(A.g0, A.g_dtype, off, rg);
        radix_fetch<S>(A.g1, A.g_dtype, off, rh);
        if (item == item0) fused_load_weights<EC, S::NW>(A, head, w_lds);
        K k{A, it, w_lds, dw_mine, exch, lane, wave, fl};
        radix_commit<S>(ry, A.in_dtype, A.tab.kappa, k.Y);
        radix_commit<S>(rb, A.in_dtype, A.tab.b_scale, k.B);
        radix_commit<S>(rg, A.g_dtype, 1.0f, k.G);
        radix_commit<S>(rh, A.g_dtype, 1.0f, k.P);
#pragma unroll
        for (int r = 0; r < S::R; ++r)
#pragma unroll
            for (int f = 0; f < S::F; ++f) k.P[r][f] = fmaf(A.tab.om, k.G[r][f], k.P[r][f]);   // p = (1-m) g + h
        if (__any(exists != (1u << S::R) - 1u)) {   // rows that do not exist must add nothing to dW
#pragma unroll
            for (int r = 0; r < S::R; ++r) {
                const bool dead = !((exists >> r) & 1u);
#pragma unroll
                for (int f = 0; f < S::F; ++f) {
                    k.Y[r][f] = dead ? 0.f : k.Y[r][f]; k.B[r][f] = dead ? 0.f : k.B[r][f];
                    k.G[r][f] = dead ? 0.f : k.G[r][f]; k.P[r][f] = dead ? 0.f : k.P[r][f];
                }
            }
        }
        __syncthreads();
        k.run();
    } while (LOOP && (item += gridDim.x) < A.total_items);
    __syncthreads();
    // one partial row per workgroup and stage; the workgroup of item i owns slot (i / n_head, head i % n_head)
    float* prow = A.dw_partials + (int64_t)(item0 / A.n_head) * A.n_stages * (2 * A.E);
    for (int k = threadIdx.x; k < A.n_stages * 2 * EC; k += 64 * S::NW) {
        const int st = k / (2 * EC), rem = k - st * 2 * EC, half = rem / EC, f = rem - half * EC;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < S::NW; ++w) sum += dw_all[w * dw_stride + st * 2 * EC + rem];
        prow[(int64_t)st * (2 * A.E) + (int64_t)half * A.E + (int64_t)head * EC + f] = sum;
    }
}

}  // namespace ncn
