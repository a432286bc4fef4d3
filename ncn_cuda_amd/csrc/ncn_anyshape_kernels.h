// Register-tile stage kernels for group sizes and head widths that are no powers of two.
//
// Same decomposition and step arithmetic as ncn_stage_kernels.h (see there for the formulas and their reference
// citations), with a geometry that is chosen per launch instead of compiled in: a lane holds an R x F tile (R = 2..5
// rows, F = 3..5 features), a row is spread over LF = 2^lf_log2 lanes and a group over
// LR = 2^lr_log2 row lanes, so that R * LR covers n_cache rows and F * LF the head's features with little padding
// (any_tile() in ncn_launch.h; 5 rows of 40 features: R = 3, F = 5, LF = 8, LR = 2, one row of six padded).  Padded
// features have zero weights and zero gradients, which stay zero; padded rows have zero gradients, which stay zero, and
// never are a pivot.  Where a head is a whole number of lanes, a lane holds F adjacent features, which one instruction of up
// to four words moves (AnyFrag); elsewhere the feature of register f is f * LF + (lane % LF), one word at a time, because a
// lane's F adjacent features would reach past the head.
//
// What bounds it: vector issue, as for the shapes of powers of two; the levels of the cross-lane sums are taken under
// wave-uniform branches because LF and LR are not known at compile time.  One lane per row with the state in LDS (the
// generic kernels, which still take what fits no tile, scalars outside the scaled state and m < 0.85) leaves three quarters of
// the time to LDS traffic and its barriers.
// 16 x 1005 x 160 float32, groups of 5 rows, heads of 40: forward 113 -> 15.5 us, backward 519 -> 26.3 us per stage.
#pragma once
#include <type_traits>

#include "ncn_stage_kernels.h"

namespace ncn {

// Sums across lanes, the levels (lane bits) known at run time and the same for the wave: over the 2^hi lanes of a row ..
template <int N>
__device__ __forceinline__ void any_sum_rows(float (&v)[N], int hi) {
#define NCN_LEVEL(S)                                                    \
    _Pragma("unroll") for (int k = 0; k < N; ++k) v[k] += lane_xor<S, true>(v[k]);
    if (hi > 0) {
        NCN_LEVEL(1)
        if (hi > 1) {
            NCN_LEVEL(2)
            if (hi > 2) {
                NCN_LEVEL(4)
                if (hi > 3) {
                    NCN_LEVEL(8)
                    if (hi > 4) { NCN_LEVEL(16) }
                }
            }
        }
    }
}
// .. and over the lanes that differ in the bits lo .. hi-1
template <int N>
__device__ __forceinline__ void any_sum_span(float (&v)[N], int lo, int hi) {
    if (lo >= hi) return;
    if (lo <= 0) { NCN_LEVEL(1) }
    if (lo <= 1 && hi > 1) { NCN_LEVEL(2) }
    if (lo <= 2 && hi > 2) { NCN_LEVEL(4) }
    if (lo <= 3 && hi > 3) { NCN_LEVEL(8) }
    if (lo <= 4 && hi > 4) { NCN_LEVEL(16) }
    if (lo <= 5 && hi > 5) { NCN_LEVEL(32) }
#undef NCN_LEVEL
}

// One wave tile of a launch: where this lane's rows and features are.
template <int R, int F, bool LENGTHS>
struct AnyLane {
    int lfl, lrl, fl, rl, gw;   // log2 of lanes per row and row lanes per group; this lane's place
    int head_dim;
    bool whole;                 // head_dim is a multiple of F: register f of lane fl is feature fl * F + f, else (f << lfl) + fl
    int64_t entry;              // element offset of the tile's batch entry (wave-uniform)
    uint32_t row[R];            // elements from there to the row's head slice: 32-bit offsets from a scalar base
    int live;                   // live rows of the lane's group, -1 past the last group
    __device__ __forceinline__ void place(const StageArgs& A, int lane) {
        lfl = (A.any_tile >> 16) & 0xff;
        lrl = A.any_tile >> 24;
        fl = lane & ((1 << lfl) - 1);
        rl = (lane >> lfl) & ((1 << lrl) - 1);
        gw = lane >> (lfl + lrl);
        head_dim = A.head_dim;
        whole = head_dim % F == 0;
    }
    // feature of register f, clamped into the head, and whether it exists: made again where they are needed, for they would
    // take 2 F registers across the steps
    __device__ __forceinline__ int feat0() const { return min(fl * F, head_dim - F); }   // first of a lane's features, when whole
    __device__ __forceinline__ int feat(int f) const { return whole ? feat0() + f : min((f << lfl) + fl, head_dim - 1); }
    __device__ __forceinline__ bool has(int f) const { return whole ? fl * F < head_dim : (f << lfl) + fl < head_dim; }
    __device__ __forceinline__ void rows(const StageArgs& A, uint32_t t, int head) {
        const uint32_t b = t / A.tiles_per_inst;
        const uint32_t group = (t - b * A.tiles_per_inst) * (64u >> (lfl + lrl)) + gw;
        const bool valid = group < A.groups;
        live = !valid ? -1 : LENGTHS ? live_rows(A, b, group) : A.n_cache;
        entry = (int64_t)b * A.N * A.E;
        // slot_position() of every row, with one branch on the kind of grouping around them all: a branch per row would wait
        // for the arguments, and behind a table for memory, row by row
        const uint32_t g = valid ? group : 0u, n = A.n_cache;
        uint32_t pos[R];
        if (A.table) {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) pos[rr] = A.table[(int64_t)g * n + min((uint32_t)(rl * R + rr), n - 1u)];
#pragma unroll
            for (int rr = 0; rr < R; ++rr) pos[rr] = (uint32_t)max(0, min((int32_t)pos[rr], (int32_t)A.N - 1));
        } else if (A.radix_stride) {
            const uint32_t s = A.radix_stride, hi = g / s;
#pragma unroll
            for (int rr = 0; rr < R; ++rr) pos[rr] = (hi * n + min((uint32_t)(rl * R + rr), n - 1u)) * s + (g - hi * s);
        } else {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) {
                const uint32_t slot = min((uint32_t)(rl * R + rr), n - 1u);
                pos[rr] = stage_block(A, g, slot) * n + slot;
            }
        }
#pragma unroll
        for (int rr = 0; rr < R; ++rr) row[rr] = pos[rr] * (uint32_t)A.E + head * A.head_dim;
    }
    // Between the loads and the stores of a tile: the compiler would otherwise keep the R x F element offsets it made for
    // the loads in registers across the steps instead of making them again.
    __device__ __forceinline__ void forget_offsets() {
#pragma unroll
        for (int rr = 0; rr < R; ++rr) asm volatile("" : "+v"(row[rr]));
        asm volatile("" : "+v"(fl));
    }
    // the row is one of the group's: it takes part in the steps (run) or lies past a context length (pass)
    __device__ __forceinline__ bool run(int rr) const { return rl * R + rr < live; }
    __device__ __forceinline__ bool pass(const StageArgs& A, int rr) const {
        return live >= 0 && rl * R + rr >= live && rl * R + rr < A.n_cache;
    }
};

template <typename T>
__device__ __forceinline__ T* any_at(T* entry, uint32_t elem) {
    // (by way of an integer the address would lose its address space, and every load and store become a flat one)
    return reinterpret_cast<T*>(const_cast<char*>(reinterpret_cast<const char*>(entry)) + (uint32_t)(elem * sizeof(T)));
}

// The weights of a lane times gamma, zero in features that do not exist.  All requested before any is waited for.
template <int R, int F, bool LENGTHS>
__device__ __forceinline__ void any_weights(const StageArgs& A, const AnyLane<R, F, LENGTHS>& L, int head, float (&wi)[F], float (&wj)[F]) {
    const int64_t at = (int64_t)head * A.head_dim;
    if (A.w_bf16) {
        const uint16_t *i = static_cast<const uint16_t*>(A.W) + at, *j = i + A.E;
        uint32_t ri[F], rj[F];
#pragma unroll
        for (int f = 0; f < F; ++f) { ri[f] = i[L.feat(f)]; rj[f] = j[L.feat(f)]; }
#pragma unroll
        for (int f = 0; f < F; ++f) { wi[f] = bf16_to_f32(ri[f]); wj[f] = bf16_to_f32(rj[f]); }
    } else {
        const float *i = static_cast<const float*>(A.W) + at, *j = i + A.E;
#pragma unroll
        for (int f = 0; f < F; ++f) { wi[f] = i[L.feat(f)]; wj[f] = j[L.feat(f)]; }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        wi[f] = L.has(f) ? A.tab.gamma * wi[f] : 0.f;
        wj[f] = L.has(f) ? A.tab.gamma * wj[f] : 0.f;
    }
}

// A lane's F adjacent features of a row, at any element: loads and stores of up to four words where the head is a whole number of
// lanes.  Launches on x[16, 1005, 160], heads of 40, groups of 5, float32, us: one word at a time by flat instructions, over eight
// rows each, with the weights one latency after the other and a loop over tiles: forward 17.3, backward 33.3 (20 of them without
// its steps); weights behind the tile and no loop 17.0 and 30.7; adjacent features 15.8 and 28.3; global instructions 15.5 and 26.3.
template <typename T, int F>
struct __attribute__((packed, aligned(sizeof(T)))) AnyFrag {
    T v[F];
};

// The loads of a tile, as raw words (converted by any_finish), so that those of all arrays of a tile are under way together.
template <int R, int F, bool LENGTHS>
__device__ __forceinline__ void any_issue(const void* base, int dtype, const AnyLane<R, F, LENGTHS>& L, float (&v)[R][F]) {
    if (L.whole) {
        const uint32_t f0 = L.feat0();
        if (dtype == NCN_F32) {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) {
                const auto q = *reinterpret_cast<const AnyFrag<float, F>*>(any_at(static_cast<const float*>(base) + L.entry, L.row[rr] + f0));
#pragma unroll
                for (int f = 0; f < F; ++f) v[rr][f] = q.v[f];
            }
        } else {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) {
                const auto q = *reinterpret_cast<const AnyFrag<uint16_t, F>*>(any_at(static_cast<const uint16_t*>(base) + L.entry, L.row[rr] + f0));
#pragma unroll
                for (int f = 0; f < F; ++f) v[rr][f] = __uint_as_float(q.v[f]);
            }
        }
    } else if (dtype == NCN_F32) {
#pragma unroll
        for (int rr = 0; rr < R; ++rr)
#pragma unroll
            for (int f = 0; f < F; ++f) v[rr][f] = *any_at(static_cast<const float*>(base) + L.entry, L.row[rr] + L.feat(f));
    } else {
#pragma unroll
        for (int rr = 0; rr < R; ++rr)
#pragma unroll
            for (int f = 0; f < F; ++f)
                v[rr][f] = __uint_as_float(*any_at(static_cast<const uint16_t*>(base) + L.entry, L.row[rr] + L.feat(f)));
    }
}
template <int R, int F>
__device__ __forceinline__ void any_finish(int dtype, float (&v)[R][F]) {
    if (dtype == NCN_F32) return;
#pragma unroll
    for (int rr = 0; rr < R; ++rr)
#pragma unroll
        for (int f = 0; f < F; ++f) v[rr][f] = __uint_as_float(__float_as_uint(v[rr][f]) << 16);
}
// Rows that do not run become zero, features that do not exist `missing`: zero, or for x (y), which every row sum multiplies,
// any other number.  Their weights are zero, so they add nothing to a sum; but an infinite sum times zero would be NaN, which
// the next sum spreads over the row, where times one it saturates the activation as it does in the features that exist.
template <int R, int F, bool LENGTHS>
__device__ __forceinline__ void any_fill_padding(const AnyLane<R, F, LENGTHS>& L, float (&v)[R][F], float missing = 0.f) {
#pragma unroll
    for (int rr = 0; rr < R; ++rr)
#pragma unroll
        for (int f = 0; f < F; ++f) v[rr][f] = !L.run(rr) ? 0.f : L.has(f) ? v[rr][f] : missing;
}
// for a tile whose steps are undone, which multiplies by 1/m each time: where (1/m)^n would leave the range of float32, zero
__device__ __forceinline__ float any_missing_undone(const StepTable& S) { return S.m_pow_n > 1e-30f ? 1.f : 0.f; }
// both arrays of a pair, the rows that take part in the steps (DEAD = false) or those that pass through
template <bool DEAD, int R, int F, bool LENGTHS>
__device__ __forceinline__ void any_store(const StageArgs& A, const AnyLane<R, F, LENGTHS>& L, void* base0, void* base1, int dtype,
                                          const float (&p)[R][F], const float (&q)[R][F]) {
    if (L.whole) {
        const uint32_t f0 = L.feat0();
#pragma unroll
        for (int rr = 0; rr < R; ++rr)
            if ((DEAD ? L.pass(A, rr) : L.run(rr)) && L.has(0)) {
                const uint32_t at = L.row[rr] + f0;
                if (dtype == NCN_F32) {
                    AnyFrag<float, F> fp, fq;
#pragma unroll
                    for (int f = 0; f < F; ++f) { fp.v[f] = p[rr][f]; fq.v[f] = q[rr][f]; }
                    *reinterpret_cast<AnyFrag<float, F>*>(any_at(static_cast<float*>(base0) + L.entry, at)) = fp;
                    *reinterpret_cast<AnyFrag<float, F>*>(any_at(static_cast<float*>(base1) + L.entry, at)) = fq;
                } else {
                    AnyFrag<uint16_t, F> fp, fq;
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        const uint32_t pq = pack_bf16x2(p[rr][f], q[rr][f]);
                        fp.v[f] = (uint16_t)pq;
                        fq.v[f] = (uint16_t)(pq >> 16);
                    }
                    *reinterpret_cast<AnyFrag<uint16_t, F>*>(any_at(static_cast<uint16_t*>(base0) + L.entry, at)) = fp;
                    *reinterpret_cast<AnyFrag<uint16_t, F>*>(any_at(static_cast<uint16_t*>(base1) + L.entry, at)) = fq;
                }
            }
        return;
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr)
        if (DEAD ? L.pass(A, rr) : L.run(rr)) {
#pragma unroll
            for (int f = 0; f < F; ++f)
                if (L.has(f)) {
                    const uint32_t at = L.row[rr] + L.feat(f);
                    if (dtype == NCN_F32) {
                        *any_at(static_cast<float*>(base0) + L.entry, at) = p[rr][f];
                        *any_at(static_cast<float*>(base1) + L.entry, at) = q[rr][f];
                    } else {
                        const uint32_t pq = pack_bf16x2(p[rr][f], q[rr][f]);
                        *any_at(static_cast<uint16_t*>(base0) + L.entry, at) = (uint16_t)pq;
                        *any_at(static_cast<uint16_t*>(base1) + L.entry, at) = (uint16_t)(pq >> 16);
                    }
                }
        }
}

// The pivot row's fragment for every lane of its group (row lane jo holds it), through wave-private LDS slots; a wave's
// LDS operations complete in order, so no barrier.
template <int F>
__device__ __forceinline__ void any_broadcast(const float (&v)[F], float (&out)[F], bool many, int src, int lane, float* slots) {
    if (!many) {
#pragma unroll
        for (int f = 0; f < F; ++f) out[f] = v[f];
        return;
    }
#pragma unroll
    for (int f = 0; f < F; ++f) slots[f * 64 + lane] = v[f];
#pragma unroll
    for (int f = 0; f < F; ++f) out[f] = slots[f * 64 + src];
}

template <bool PRIORITY, int R, int F>
__device__ __forceinline__ void any_row_sums(const float (&x)[R][F], const float (&wi)[F], float e, int lfl, float (&c)[R]) {
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        c[rr] = e;
#pragma unroll
        for (int f = 0; f < F; ++f) c[rr] = fmaf(x[rr][f], wi[f], c[rr]);
    }
    issue_first<PRIORITY>();   // (the wave stays at high priority)
    any_sum_rows<R>(c, lfl);
}

// f(0), f(1), .., f(N-1) with the index a compile-time constant.  (An unrolled loop over the pivot rows is not enough: with
// a step that may be skipped the compiler gives the tile a place in scratch memory before it unrolls.)
template <int N, int I = 0, typename Fn>
__device__ __forceinline__ void for_each_row(const Fn& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        for_each_row<N, I + 1>(f);
    }
}

#define NCN_ANY_PROLOGUE                                                                        \
    const int lane = threadIdx.x & 63;                                                          \
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);                          \
    const uint32_t gwave = blockIdx.x * kWavesPerBlock + wave;                                  \
    const int head = gwave % A.n_head;                                                          \
    const uint32_t tile_step = gridDim.x * kWavesPerBlock / A.n_head;                           \
    __shared__ float bcast_lds[kWavesPerBlock * F * 64];                                        \
    float* slots = bcast_lds + wave * F * 64;                                                   \
    AnyLane<R, F, LENGTHS> L;                                                                            \
    L.place(A, lane);                                                                           \
    const int lr = 1 << L.lrl;                                                                  \
    const StepTable& S = A.tab;                                                                 \
    float wi[F], wj[F];

constexpr int kAnyPriorityRows = 12;

// INVERSE = false: x, xa -> y, ya (optional float32 copies);  true: y, ya -> x, xa
// PRIORITY: exp2 at high priority, one constant in a vector register (issue_first, in_vector_register), for launches with
// kAnyPriorityRows and more to a group and no lengths.  us, without : with (x[24, 8192, ~256] float32, forward / inverse): groups of 48,
// heads of 20 602 : 525 / 597 : 526, of 24, 12 386 : 357 / 366 : 347, of 20, 40 345 : 326 / 338 : 321, of 12, 48 208 : 201 / 206 : 192; of 10,
// 40 218 : 235 / 212 : 228, of 5, 5 430 : 430 / 452 : 470, of 3, 7 the same.  With lengths 381 : 366 / 376 : 358, 265 : 272 / 275 : 273, 244 : 242 /
// 242 : 233, 168 : 177 / 176 : 176, of 5, 5 601 : 597 / 584 : 625, of 3, 7 467 : 497 / 487 : 486; so not there, nor with other activations.
template <int R, int F, bool TANH_ONLY, bool INVERSE, bool LENGTHS, bool PRIORITY>
__global__ void __launch_bounds__(kBlockThreads, R * F <= 16 ? 4 : R * F <= 20 ? 3 : 2) any_forward_kernel(const StageArgs A) {
    NCN_ANY_PROLOGUE
    for (uint32_t t = gwave / A.n_head; t < A.total_tiles; t += tile_step) {
        L.rows(A, t, head);
        float x[R][F], a[R][F];
        any_issue(A.in0, A.in_dtype, L, x);
        any_issue(A.in1, A.in_dtype, L, a);
        if constexpr (!LENGTHS) any_weights(A, L, head, wi, wj);   // behind the tile's own loads: one latency, not two
        any_finish(A.in_dtype, x);
        any_finish(A.in_dtype, a);
        if constexpr (LENGTHS) {
            if (__any(L.live >= 0 && L.live < (int)A.n_cache)) {   // rows past a context length pass through
                any_store<true>(A, L, A.out0, A.out1, A.out_dtype, x, a);
                if (!INVERSE && A.aux0) any_store<true>(A, L, A.aux0, A.aux1, NCN_F32, x, a);
            }
            // after those stores, beside which the weights would take 10 to 20 registers and a SIMD hold four or five waves instead
            // of six or seven: x[1559, 48, 40] bfloat16 with lengths, groups of 16, heads of 20, sigmoid, forward 44.7 us, here 37.8
            any_weights(A, L, head, wi, wj);
        }
        any_fill_padding(L, x, INVERSE ? any_missing_undone(S) : 1.f);
        any_fill_padding(L, a);
        scale_tile<R, F>(x, a, S.kappa, INVERSE ? S.b_scale : S.a_scale);
        const float keep = PRIORITY ? in_vector_register(INVERSE ? S.im : S.m) : INVERSE ? S.im : S.m;   // read twice per element and step
#pragma unroll 1
        for (int k = 0; k < lr; ++k) {
            const int jo = INVERSE ? lr - 1 - k : k;
            const int src = (lane & ~((lr - 1) << L.lfl)) | (jo << L.lfl);
            for_each_row<R>([&](auto q) __attribute__((always_inline)) {
                constexpr int jr = INVERSE ? R - 1 - q.value : q.value;
                if (jo * R + jr >= (LENGTHS ? L.live : A.n_cache)) return;   // LENGTHS: the lanes of a group agree
                if constexpr (INVERSE) {
#pragma unroll
                    for (int rr = 0; rr < R; ++rr)
#pragma unroll
                        for (int f = 0; f < F; ++f) x[rr][f] = fmaf(keep, x[rr][f], -a[rr][f]);
                }
                float xj[F], c[R];
                any_broadcast<F>(x[jr], xj, lr > 1, src, lane, slots);
                any_row_sums<PRIORITY, R, F>(x, wi, dot_chain<F>(xj, wj), L.lfl, c);
                if constexpr (TANH_ONLY) {
                    float r[R][F];
                    sigmoids(0, x, c, xj, r);
                    issue_with_others<PRIORITY>();
#pragma unroll
                    for (int rr = 0; rr < R; ++rr)
#pragma unroll
                        for (int f = 0; f < F; ++f) {
                            a[rr][f] = fmaf(INVERSE ? S.bk1 : S.m2k2, r[rr][f], fmaf(keep, a[rr][f], INVERSE ? S.bk0 : S.k2));
                            if constexpr (!INVERSE) x[rr][f] = fmaf(keep, x[rr][f], a[rr][f]);
                        }
                } else {
#pragma unroll
                    for (int rr = 0; rr < R; ++rr)
#pragma unroll
                        for (int f = 0; f < F; ++f) {
                            float Fv, w;
                            act_Fw(fmaf(c[rr], xj[f], x[rr][f]), S.activation, Fv, w);
                            a[rr][f] = fmaf(INVERSE ? S.bk0 : S.k2, Fv, keep * a[rr][f]);
                            if constexpr (!INVERSE) x[rr][f] = fmaf(keep, x[rr][f], a[rr][f]);
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        L.forget_offsets();
        scale_tile<R, F>(x, a, S.inv_kappa, INVERSE ? S.inv_b_scale : S.inv_a_scale);
        any_store<false>(A, L, A.out0, A.out1, A.out_dtype, x, a);
        if (!INVERSE && A.aux0) any_store<false>(A, L, A.aux0, A.aux1, NCN_F32, x, a);
    }
}

// LOOP = false: launches with a wave for every tile (tiles of up to 15 elements, whose loop builds need 16 to 24 registers more;
// larger ones spill without it).  Three rows of five features run three waves per SIMD: at four, 16 registers spill and a backward
// launch of the figures above takes 29.3 us.
template <int R, int F, bool TANH_ONLY, bool LENGTHS, bool LOOP>
__global__ void __launch_bounds__(kBlockThreads, R * F <= (LOOP ? 10 : 12) ? 4 : R * F <= 16 ? 3 : 2) any_backward_kernel(const StageArgs A) {
    NCN_ANY_PROLOGUE
    constexpr bool kKuW = LOOP || R * F <= 10;   // ku Wi' kept beside the weights, where there are registers for it
    float dwi[F], dwj[F], wiku[kKuW ? F : 1];
#pragma unroll
    for (int f = 0; f < F; ++f) dwi[f] = dwj[f] = 0.f;
    auto weights = [&]() {
        any_weights(A, L, head, wi, wj);
        if constexpr (kKuW) {
#pragma unroll
            for (int f = 0; f < F; ++f) wiku[f] = S.ku * wi[f];
        }
    };
    if constexpr (LOOP) weights();
    uint32_t t = gwave / A.n_head;
    if (t < A.total_tiles) do {
        L.rows(A, t, head);
        float Y[R][F], B[R][F], G[R][F], P[R][F];
        any_issue(A.in0, A.in_dtype, L, Y);
        any_issue(A.in1, A.in_dtype, L, B);
        any_issue(A.g0, A.g_dtype, L, G);
        if (A.g1) {
            any_issue(A.g1, A.g_dtype, L, P);
        } else {
#pragma unroll
            for (int rr = 0; rr < R; ++rr)
#pragma unroll
                for (int f = 0; f < F; ++f) P[rr][f] = 0.f;
        }
        if constexpr (!LOOP) weights();   // behind the tile's own loads: one latency, not two
        any_finish(A.in_dtype, Y);
        any_finish(A.in_dtype, B);
        any_finish(A.g_dtype, G);
        if (A.g1) any_finish(A.g_dtype, P);
        if (LENGTHS) {
            any_store<true>(A, L, A.out0, A.out1, A.out_dtype, G, P);
            if (A.aux0) any_store<true>(A, L, A.aux0, A.aux1, NCN_F32, Y, B);
        }
        any_fill_padding(L, Y, any_missing_undone(S));
        any_fill_padding(L, B);
        any_fill_padding(L, G);
        any_fill_padding(L, P);
        // as if the steps that a group cut by a context length skips had been done: G, P carry m^-t
        const float isc = LENGTHS && L.live < A.n_cache ? pow_steps(S.im, A.n_cache - L.live) : 1.0f;
#pragma unroll
        for (int rr = 0; rr < R; ++rr)
#pragma unroll
            for (int f = 0; f < F; ++f) {
                Y[rr][f] *= S.kappa;
                B[rr][f] *= S.b_scale;
                P[rr][f] = isc * fmaf(S.om, G[rr][f], P[rr][f]);   // h -> p
                G[rr][f] *= isc;
            }
#pragma unroll 1
        for (int jo = lr - 1; jo >= 0; --jo) {
            const float selku = L.rl == jo ? S.ku : 0.f;   // this lane holds the pivot row
            const int src = (lane & ~((lr - 1) << L.lfl)) | (jo << L.lfl);
            for_each_row<R>([&](auto q) __attribute__((always_inline)) {
                constexpr int jr = R - 1 - q.value;
                const int j = jo * R + jr;
                if (j >= (LENGTHS ? L.live : A.n_cache)) return;
                const float krho = S.krho[A.n_cache - 1 - j];
#pragma unroll
                for (int rr = 0; rr < R; ++rr)
#pragma unroll
                    for (int f = 0; f < F; ++f) Y[rr][f] = fmaf(S.im, Y[rr][f], -B[rr][f]);
                float xj[F], c[R], rh[R], v[F];
                any_broadcast<F>(Y[jr], xj, lr > 1, src, lane, slots);
                any_row_sums<TANH_ONLY, R, F>(Y, wi, dot_chain<F>(xj, wj), L.lfl, c);
#pragma unroll
                for (int f = 0; f < F; ++f) v[f] = 0.f;
#pragma unroll
                for (int rr = 0; rr < R; ++rr) {   // exp2 and reciprocals of one row at a time: see backward_core
                    float r[1][F];
                    if constexpr (TANH_ONLY) {
                        if (rr > 0) issue_first();
                        sigmoids(rr, Y, c, xj, r);
                        issue_with_others();
                    }
                    rh[rr] = 0.f;
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        float w;
                        if constexpr (TANH_ONLY) {
                            B[rr][f] = fmaf(S.bk1, r[0][f], fmaf(S.im, B[rr][f], S.bk0));
                            w = fmaf(-r[0][f], r[0][f], r[0][f]);
                        } else {
                            float Fv;
                            act_Fw(fmaf(c[rr], xj[f], Y[rr][f]), S.activation, Fv, w);
                            B[rr][f] = fmaf(S.bk0, Fv, S.im * B[rr][f]);
                        }
                        const float U = P[rr][f] * w;
                        rh[rr] = fmaf(U, xj[f], rh[rr]);
                        v[f] = fmaf(c[rr], U, v[f]);
                        G[rr][f] = fmaf(S.ku, U, G[rr][f]);
                    }
                }
                issue_first<TANH_ONLY>();
                any_sum_rows<R>(rh, L.lfl);
                issue_with_others<TANH_ONLY>();
                float rhosum = 0.f;
#pragma unroll
                for (int rr = 0; rr < R; ++rr) {
                    const float rho_w = krho * rh[rr];
                    const float rho_ku = kKuW ? rh[rr] : S.ku * rh[rr];
                    rhosum += rh[rr];
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        dwi[f] = fmaf(rho_w, Y[rr][f], dwi[f]);
                        G[rr][f] = fmaf(rho_ku, kKuW ? wiku[f] : wi[f], G[rr][f]);
                        if (rr != jr) P[rr][f] = fmaf(S.om, G[rr][f], P[rr][f]);
                    }
                }
                const float rhosum_w = krho * rhosum;
                float s[F];
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    dwj[f] = fmaf(rhosum_w, xj[f], dwj[f]);
                    s[f] = fmaf(rhosum, wj[f], v[f]);
                }
                issue_first<TANH_ONLY>();
                any_sum_span<F>(s, L.lfl, L.lfl + L.lrl);   // over the group's row lanes
                issue_with_others<TANH_ONLY>();
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    G[jr][f] = fmaf(selku, s[f], G[jr][f]);
                    P[jr][f] = fmaf(S.om, G[jr][f], P[jr][f]);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
#pragma unroll
        for (int rr = 0; rr < R; ++rr)
#pragma unroll
            for (int f = 0; f < F; ++f) {
                G[rr][f] *= S.m_pow_n;
                P[rr][f] = fmaf(P[rr][f], S.m_pow_n, -S.om * G[rr][f]);   // back to h = p - (1-m) g
            }
        L.forget_offsets();
        any_store<false>(A, L, A.out0, A.out1, A.out_dtype, G, P);
        if (A.aux0) {
            scale_tile<R, F>(Y, B, S.inv_kappa, S.inv_b_scale);
            any_store<false>(A, L, A.aux0, A.aux1, NCN_F32, Y, B);
        }
    } while (LOOP && (t += tile_step) < A.total_tiles);
    // dW: lanes holding the same features -> one value; this wave owns slot (gwave / n_head, head)
    any_sum_span<F>(dwi, L.lfl, 6);
    any_sum_span<F>(dwj, L.lfl, 6);
    if (lane < (1 << L.lfl)) {
        float* out = A.dw_partials + (int64_t)(gwave / A.n_head) * (2 * A.E) + (int64_t)head * A.head_dim;
#pragma unroll
        for (int f = 0; f < F; ++f)
            if (L.has(f)) {
                out[L.feat(f)] = dwi[f];
                out[A.E + L.feat(f)] = dwj[f];
            }
    }
}
#undef NCN_ANY_PROLOGUE

}  // namespace ncn
