// Multi-stage passes for groups of FOUR rows under the stride permutation, whole groups in the registers of a lane.
//
// Each lane holds a 4 x 4 tile: the four rows of its group times four features, so that the LF = EC/4 lanes of a row hold
// a group, no step needs another lane's rows (the pivot row is always in the lane itself) and a wave carries 64/LF groups,
// one tile per wave and window.  The rows stay in registers from the window's load to its store; between two stages slot
// o of a group moves to the group o * (difference of the strides) further on, and slots 1 to 3 change hands through LDS
// (slot 0 never moves).  A wave starts on its groups when its own rows have come and stores them when they are done:
// only the exchanges wait for the whole workgroup.  (The kernels of ncn_fused_kernels.h, which these replace but for context
// lengths, keep every row in LDS, spread a group over two lanes per feature and pass the pivot row between them.)
//
// x[64, 2048, 128] bfloat16, groups of 4, 6 stages in two passes: forward passes 109 + 128 -> 94 + 115 us, backward 268 + 239 ->
// 227 + 202; x[32, 1024, 128] float32, 5 stages: 37 + 23 -> 35 + 21 and 62 + 51 -> 55 + 44.  With issue_first (ncn_device.h) the larger
// ones take 80 + 102 and 168 + 153: without loads and stores 67 + 78 and 155 + 136, without steps 43 + 69 and 86 + 98.
#pragma once
#include "ncn_fused_kernels.h"

namespace ncn {

constexpr int kQuadF = 4;              // features per lane
// Waves per workgroup: windows of 2048 / EC groups forward, 1024 / EC backward.  (Backward windows of 8 waves, with
// half the halo, have all waves of a workgroup wait for each other: 207 + 185 us the passes of x[64, 2048, 128] above against 157 + 145, 46 + 56 those
// of x[32, 1024, 128] against 39 + 48.)
constexpr int kQuadWavesFwd = 8, kQuadWavesBwd = 4;
constexpr int quad_groups(int ec, int waves) { return waves * (64 * kQuadF / ec); }   // groups of the largest window
constexpr size_t quad_lds_bytes(int ec, int waves, bool backward) {
    return ((size_t)2 * 3 * quad_groups(ec, waves) + (backward ? 2 * kFusedMaxStages + 2 * waves : 0)) * ec * sizeof(float);
}

// Lane's row fragments to the LDS place of its window position, slots 1 to 3 (slot 0 stays).
template <int EC, int W>
__device__ __forceinline__ void quad_put(float* buf, uint32_t q, int fl, const float (&v)[4][kQuadF]) {
#pragma unroll
    for (int o = 1; o < 4; ++o) lds_store_frag<kQuadF>(buf + ((o - 1) * W + q) * EC + fl * kQuadF, v[o]);
}
template <int EC, int W>
__device__ __forceinline__ void quad_get(const float* buf, const uint32_t (&from)[4], int fl, float (&v)[4][kQuadF]) {
#pragma unroll
    for (int o = 1; o < 4; ++o) lds_load_frag<kQuadF>(buf + ((o - 1) * W + from[o]) * EC + fl * kQuadF, v[o]);
}
// Window positions that hold the slots of position q's group in the stage with stride `to`, after one with `at`.
template <int W>
__device__ __forceinline__ void quad_partners(const FusedArgs& A, uint32_t q, int at, int to, uint32_t (&from)[4]) {
    if (A.closed) {
        uint32_t step = (uint32_t)(to - at) + (to < at ? A.ring : 0u);   // on the ring
#pragma unroll
        for (uint32_t o = 1; o < 4; ++o) from[o] = q < A.window ? ring_wrap(A, q, o * step) : q;
    } else {
#pragma unroll
        for (int o = 1; o < 4; ++o) from[o] = (uint32_t)max(0, min((int)q + o * (to - at), W - 1));
    }
}
// Row offsets of the lane's group as a stage with stride `ss` has it.
template <int EC>
__device__ __forceinline__ void quad_offsets(const FusedArgs& A, const FusedItem& it, uint32_t q, int ss, int fl, int64_t (&off)[4]) {
#pragma unroll
    for (uint32_t o = 0; o < 4; ++o) {
        const uint32_t at = A.closed ? ring_wrap(A, q, o * (uint32_t)ss) : q + o * (uint32_t)ss;
        off[o] = fused_row_offset<4, false>(A, it, at * 4u + o) + fl * kQuadF;
    }
}

// A lane's weights of stage `st`: requested (raw, no branch on the type: see issue_w), and as float32 times gamma.  Straight from
// memory a stage ahead, so that no wave has to wait for another's loads before it starts.
__device__ __forceinline__ void quad_issue_w(const FusedArgs& A, int st, int at, float (&wi)[kQuadF], float (&wj)[kQuadF]) {
    const int log2_size = A.w_bf16 ? 1 : 2, second = A.w_bf16 ? 0 : 8;
    const char* const wi_at = static_cast<const char*>(A.W[st]) + ((int64_t)at << log2_size);
    const char* const wj_at = wi_at + (A.E << log2_size);
    const float2 i0 = *reinterpret_cast<const float2*>(wi_at), i1 = *reinterpret_cast<const float2*>(wi_at + second);
    const float2 j0 = *reinterpret_cast<const float2*>(wj_at), j1 = *reinterpret_cast<const float2*>(wj_at + second);
    wi[0] = i0.x; wi[1] = i0.y; wi[2] = i1.x; wi[3] = i1.y;
    wj[0] = j0.x; wj[1] = j0.y; wj[2] = j1.x; wj[3] = j1.y;
}
__device__ __forceinline__ void quad_finish_w(const FusedArgs& A, float (&w)[kQuadF]) {
    if (A.w_bf16) {
        const uint32_t w0 = __float_as_uint(w[0]), w1 = __float_as_uint(w[1]);
        w[0] = __uint_as_float(w0 << 16); w[1] = __uint_as_float(w0 & 0xffff0000u);
        w[2] = __uint_as_float(w1 << 16); w[3] = __uint_as_float(w1 & 0xffff0000u);
    }
#pragma unroll
    for (int f = 0; f < kQuadF; ++f) w[f] *= A.tab.gamma;
}

// forward, and with INVERSE the same passes undone (stages last to first)
template <int EC, bool TANH_ONLY, bool INVERSE, bool HEADWISE>
__global__ void __launch_bounds__(64 * kQuadWavesFwd) quad_forward_kernel(const FusedArgs A) {
    constexpr int NC = 4, R = 4, F = kQuadF, NW = kQuadWavesFwd, LF = EC / F, GPW = 64 / LF, W = NW * GPW;
    extern __shared__ float4 fused_lds4[];
    float* xs = reinterpret_cast<float*>(fused_lds4);   // [slot - 1][position][EC]
    float* as = xs + 3 * W * EC;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fl = lane % LF;
    const uint32_t q = wave * GPW + lane / LF;
    const uint32_t item = fused_deal<EC>(A, blockIdx.x);   // the launch has a workgroup for every window
    if (item >= A.total_items) return;
    const FusedItem it = fused_item<NC, EC, false>(A, item);
    const int w_at = it.head * EC + fl * F;
    float x[R][F], a[R][F], wi[F], wj[F];
    quad_issue_w(A, INVERSE ? A.n_stages - 1 : 0, w_at, wi, wj);
    {
        int64_t off[R];
        quad_offsets<EC>(A, it, min(q, A.window - 1u), A.sub_stride[INVERSE ? A.n_stages - 1 : 0], fl, off);
        issue_tile<R, F>(A.in0, A.in_dtype, off, x);
        issue_tile<R, F>(A.in1, A.in_dtype, off, a);
    }
    finish_tile<R, F>(A.in_dtype, x);
    finish_tile<R, F>(A.in_dtype, a);
    const float a_in = INVERSE ? A.tab.b_scale : A.tab.a_scale, a_out = INVERSE ? A.tab.inv_b_scale : A.tab.inv_a_scale;
#pragma unroll
    for (int o = 0; o < R; ++o)
#pragma unroll
        for (int f = 0; f < F; ++f) {
            x[o][f] *= A.tab.kappa;
            a[o][f] *= a_in;
        }
    for (int sq = 0; sq < A.n_stages; ++sq) {
        const int st = INVERSE ? A.n_stages - 1 - sq : sq;
        const int ss = A.sub_stride[st];
        const StageGroups here = stage_groups<NC>(A, ss);
        quad_finish_w(A, wi);
        quad_finish_w(A, wj);
        if (q - here.first < here.count) {   // (lanes of whole groups: every sum across lanes stays inside one)
            if constexpr (HEADWISE) {
                if (INVERSE) headwise_inverse_core<NC, EC, R, F, TANH_ONLY, false, true>(x, a, wi, wj, A.tab, lane, nullptr);
                else headwise_forward_core<NC, EC, R, F, TANH_ONLY, false, true>(x, a, wi, wj, A.tab, lane, nullptr);
            } else {
                if (INVERSE) inverse_core<NC, EC, R, F, TANH_ONLY, false, true>(x, a, wi, wj, A.tab, lane, nullptr);
                else forward_core<NC, EC, R, F, TANH_ONLY, false, true>(x, a, wi, wj, A.tab, lane, nullptr);
            }
        }
        if (sq + 1 < A.n_stages) {
            uint32_t from[4];
            const int next = INVERSE ? st - 1 : st + 1;
            quad_issue_w(A, next, w_at, wi, wj);
            quad_partners<W>(A, q, ss, A.sub_stride[next], from);
            if (sq > 0) __syncthreads();   // everyone has read the exchange before
            quad_put<EC, W>(xs, q, fl, x);
            quad_put<EC, W>(as, q, fl, a);
            __syncthreads();
            quad_get<EC, W>(xs, from, fl, x);
            quad_get<EC, W>(as, from, fl, a);
        }
    }
    if (q - it.own_lo < it.own_cnt) {   // owned rows out of the scaled form
        int64_t off[R];
        quad_offsets<EC>(A, it, q, A.sub_stride[INVERSE ? 0 : A.n_stages - 1], fl, off);
#pragma unroll
        for (int o = 0; o < R; ++o) {
            float v[F], u[F];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                v[f] = x[o][f] * A.tab.inv_kappa;
                u[f] = a[o][f] * a_out;
            }
            store_frag<F>(A.out0, A.out_dtype, off[o], true, v);
            store_frag<F>(A.out1, A.out_dtype, off[o], true, u);
            if (A.aux0) {
                store_frag<F>(A.aux0, NCN_F32, off[o], true, v);
                store_frag<F>(A.aux1, NCN_F32, off[o], true, u);
            }
        }
    }
}

// Sums each of the 8 values v[.] over the lanes of the wave that hold the same features and scatters the sums, as
// pair_scatter_sum does for 16: v[0 .. quad_scatter_left) of a lane are complete afterwards, and they are the values number
// `first` (returned) and up of the list.
template <int LF>
constexpr int quad_scatter_left() { return LF <= 8 ? 1 : LF == 16 ? 2 : 4; }
template <int LF>
__device__ __forceinline__ int quad_scatter_sum(float (&v)[8], int lane) {
    static_assert(LF == 2 || LF == 4 || LF == 8 || LF == 16 || LF == 32, "lanes per group");
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // lane bit 5
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 4]), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    int first = ((lane >> 5) & 1) * 4;
    if constexpr (LF <= 16) {   // lane bit 4
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 2]), false, false);
            v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        first += ((lane >> 4) & 1) * 2;
    }
    if constexpr (LF <= 8) {    // lane bit 3: banks 0,1 of a row keep v[0], banks 2,3 v[1] (row_ror:8 reads lane (l + 8) mod 16)
        const int lo = __float_as_int(v[0]), hi = __float_as_int(v[1]);
        const int t = __builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xF, 0x3, false);
        const int u = __builtin_amdgcn_update_dpp(lo, hi, 0x128, 0xF, 0xC, false);
        v[0] = __int_as_float(t) + __int_as_float(u);
        first += (lane >> 3) & 1;
    }
    // narrow heads: the lanes that still hold shares of the same value
    if constexpr (LF <= 4) v[0] += lane_xor<4>(v[0]);
    if constexpr (LF == 2) v[0] += lane_xor<2>(v[0]);
    return first;
}

// LOOP: workgroups walk over several windows (more windows than dW partial rows).  It spills 22 to 26 registers at four waves per SIMD, as
// builds for other activations on heads of one feature do at two (28 to 49); a wave less spills nothing and is slower: x[256, 8192, 128], 6 stages,
// heads of 8 16.2 ms : 20.9, of 32 9.0 : 8.9; sigmoid, heads of one feature, x[256, 4096, 128] 6.1 : 7.2.
template <int EC, bool TANH_ONLY, bool LOOP, bool HEADWISE>
__global__ void __launch_bounds__(64 * kQuadWavesBwd, TANH_ONLY ? 4 : 2) quad_backward_kernel(const FusedArgs A) {
    constexpr int NC = 4, R = 4, F = kQuadF, NW = kQuadWavesBwd, LF = EC / F, GPW = 64 / LF, W = NW * GPW;
    extern __shared__ float4 fused_lds4[];
    float* buf0 = reinterpret_cast<float*>(fused_lds4);   // [slot - 1][position][EC]: y and g in turns
    float* buf1 = buf0 + 3 * W * EC;                      // ya and p
    float* w_lds = buf1 + 3 * W * EC;                     // [kFusedMaxStages][2][EC]
    float* dw_lds = w_lds + kFusedMaxStages * 2 * EC;     // [wave][2][EC] of the stage
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fl = lane % LF;
    const uint32_t q = wave * GPW + lane / LF;
    const float om = 1.0f - A.tab.m;
    const uint32_t item0 = LOOP ? blockIdx.x : fused_deal<EC>(A, blockIdx.x);
    if (item0 >= A.total_items) return;
    const int head = item0 % A.n_head;   // of every window of this workgroup (gridDim.x % n_head == 0)
    // the workgroup of window i has partial row i / n_head of head i % n_head
    float* const prow = A.dw_partials + (int64_t)(item0 / A.n_head) * A.n_stages * (2 * A.E) + (int64_t)head * EC;
    fused_load_weights<EC, NW>(A, head, w_lds);   // (before the rows are asked for: no wave waits for another's rows at the barrier)
    __syncthreads();
    uint32_t item = item0;
    do {
        const FusedItem it = fused_item<NC, EC, false>(A, item);
        float Y[R][F], B[R][F], G[R][F], P[R][F];
        {
            int64_t off[R];
            quad_offsets<EC>(A, it, min(q, A.window - 1u), A.sub_stride[A.n_stages - 1], fl, off);
            issue_tile<R, F>(A.in0, A.in_dtype, off, Y);
            issue_tile<R, F>(A.in1, A.in_dtype, off, B);
            issue_tile<R, F>(A.g0, A.g_dtype, off, G);
            if (A.g1) {
                issue_tile<R, F>(A.g1, A.g_dtype, off, P);
            } else {
#pragma unroll
                for (int o = 0; o < R; ++o)
#pragma unroll
                    for (int f = 0; f < F; ++f) P[o][f] = 0.f;
            }
        }
        finish_tile<R, F>(A.in_dtype, Y);
        finish_tile<R, F>(A.in_dtype, B);
        finish_tile<R, F>(A.g_dtype, G);
        finish_tile<R, F>(A.g_dtype, P);
#pragma unroll
        for (int o = 0; o < R; ++o)
#pragma unroll
            for (int f = 0; f < F; ++f) {
                Y[o][f] *= A.tab.kappa;
                B[o][f] *= A.tab.b_scale;
                P[o][f] = fmaf(om, G[o][f], P[o][f]);   // p = (1-m) g + h
            }
        if (LOOP) __syncthreads();   // the sums of the window before are read
        for (int st = A.n_stages - 1; st >= 0; --st) {
            const int ss = A.sub_stride[st];
            const StageGroups here = stage_groups<NC>(A, ss);
            float dw[2 * F];   // this lane's share of dWi (first F) and dWj of the stage
#pragma unroll
            for (int f = 0; f < 2 * F; ++f) dw[f] = 0.f;
            if (q - here.first < here.count) {   // (lanes of whole groups: every sum across lanes stays inside one)
                float (&dwi)[F] = *reinterpret_cast<float (*)[F]>(&dw[0]);
                float (&dwj)[F] = *reinterpret_cast<float (*)[F]>(&dw[F]);
                const float own = (q - it.own_lo < it.own_cnt) ? 1.0f : 0.0f;   // unsigned: lo <= q < lo + cnt
                float wi[F], wj[F];
                lds_load_frag<F>(w_lds + st * 2 * EC + fl * F, wi);
                lds_load_frag<F>(w_lds + st * 2 * EC + EC + fl * F, wj);
                const int done = (A.n_stages - 1 - st) * NC;
                if constexpr (HEADWISE)
                    headwise_backward_core<NC, EC, R, F, true, TANH_ONLY, false, true, false, true>(Y, B, G, P, wi, wj, dwi, dwj, own, A.tab, done, lane, nullptr);
                else
                    backward_core<NC, EC, R, F, true, TANH_ONLY, false, true, false, true>(Y, B, G, P, wi, wj, dwi, dwj, own, A.tab, done, lane, nullptr);
            }
            {   // the wave's dW of the stage into its place: every lane ends up with one or more complete sums
                const int first = quad_scatter_sum<LF>(dw, lane);
                float* d = dw_lds + wave * 2 * EC + (first / F) * EC + fl * F + first % F;
                if (LF >= 8 || (lane & (LF == 4 ? 4 : 6)) == 0) {
#pragma unroll
                    for (int i = 0; i < quad_scatter_left<LF>(); ++i) d[i] = dw[i];
                }
            }
            auto sum_waves = [&]() {   // .. and the waves' sums out (the same threads each time, in a fixed order)
                for (int k = threadIdx.x; k < 2 * EC; k += 64 * NW) {
                    float sum = 0.f;
#pragma unroll
                    for (int w = 0; w < NW; ++w) sum += dw_lds[w * 2 * EC + k];
                    float* const to = prow + (int64_t)st * (2 * A.E) + (int64_t)(k / EC) * A.E + k % EC;
                    *to = LOOP && item != item0 ? *to + sum : sum;
                }
            };
            __syncthreads();   // dW is there, and everyone has read the exchange before
            if (st > 0) {
                uint32_t from[4];
                quad_partners<W>(A, q, ss, A.sub_stride[st - 1], from);
                quad_put<EC, W>(buf0, q, fl, Y);
                quad_put<EC, W>(buf1, q, fl, B);
                sum_waves();
                __syncthreads();
                quad_get<EC, W>(buf0, from, fl, Y);
                quad_get<EC, W>(buf1, from, fl, B);
                __syncthreads();
                quad_put<EC, W>(buf0, q, fl, G);
                quad_put<EC, W>(buf1, q, fl, P);
                __syncthreads();
                quad_get<EC, W>(buf0, from, fl, G);
                quad_get<EC, W>(buf1, from, fl, P);
            } else {
                sum_waves();
            }
        }
        if (q - it.own_lo < it.own_cnt) {   // owned rows: g = G m^T, h = P m^T - (1-m) g, x = xs / kappa, xa = bh / b_scale
            int64_t off[R];
            quad_offsets<EC>(A, it, q, A.sub_stride[0], fl, off);
#pragma unroll
            for (int o = 0; o < R; ++o) {
                float g[F], h[F];
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    g[f] = G[o][f] * A.scale_dn;
                    h[f] = fmaf(P[o][f], A.scale_dn, -om * g[f]);
                }
                store_frag<F>(A.out0, A.out_dtype, off[o], true, g);
                store_frag<F>(A.out1, A.out_dtype, off[o], true, h);
                if (A.aux0) {
                    float y[F], b[F];
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        y[f] = Y[o][f] * A.tab.inv_kappa;
                        b[f] = B[o][f] * A.tab.inv_b_scale;
                    }
                    store_frag<F>(A.aux0, NCN_F32, off[o], true, y);
                    store_frag<F>(A.aux1, NCN_F32, off[o], true, b);
                }
            }
        }
    } while (LOOP && (item += gridDim.x) < A.total_items);
}

}  // namespace ncn
