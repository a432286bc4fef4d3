// One-stage kernels for launches with few groups: one row fragment of 4 features per lane, and a group over as many waves
// as that takes.
//
// What bounds such a launch is the chain of its steps: with fewer waves than the chip has SIMDs nothing else issues while a
// wave waits, and every vector instruction of the 16 elements that a lane of the register tiles (ncn_stage_kernels.h) holds
// costs its latency.  A quarter of the elements per lane is a quarter of the instructions of a step; what a step then needs
// across waves is one exchange through LDS.  x[4, 256, 128], heads of 32, groups of 32 rows (128 groups, a wave each on the
// register tiles, four here), float32: forward 14.7 -> 8.2 us, backward with its dW
// reduction 37.7 -> 20.8.  (The sums across 16 and 32 lanes by v_permlane16_swap and v_permlane32_swap instead of the LDS
// crossbar: 19.9 there, but 40.2 instead of 35.6 at 1048576 elements.)
//
// A step over W > 1 waves: the waves that hold the pivot row put it into LDS, the barrier, everybody reads it.  In the
// backward the same barrier carries the previous step's share of the pivot gradient: every wave leaves the sum over its rows
// in LDS and the lanes of the pivot row add the W sums before they use that gradient again.  Both go through two
// buffers in turns: a wave that is one barrier ahead writes the buffer that nobody reads.
#pragma once
#include "ncn_stage_kernels.h"

namespace ncn {

template <int NC, int EC>
struct SplitShape {
    static constexpr int F = 4;
    static constexpr int LF = EC / F;                       // lanes per row
    static constexpr int RPW = 64 / LF;                     // rows per wave
    static constexpr int W = NC > RPW ? NC / RPW : 1;       // waves per group
    static constexpr int GPW = NC > RPW ? 1 : RPW / NC;     // groups per wave
    static constexpr int ROWS = NC / W;                     // rows of a group in a wave
    static constexpr int NW = W > 4 ? W : 4;                // waves per workgroup
    static constexpr int UNITS = NW / W;                    // units (W waves) per workgroup
    static constexpr int SLOT4 = EC / 4;                    // float4 per row
};

// Where a lane works: unit u of the launch is (wave tile u / n_head, head u % n_head).
struct SplitPlace {
    int lane, wave, fl, row, unit_in_block, wave_in_unit, head;
    uint32_t t;      // wave tile (group when W > 1)
    int live;        // live rows of the lane's group: NC, or (INDEXED) fewer behind a context length; 0: no group
    bool exists;     // the lane's group exists
    bool valid;      // .. and the lane's row is live
    int64_t off;     // element offset of the lane's fragment
};

// INDEXED builds honour a.table, a.radix_stride and a.ctx_len, as those of the register tiles do
template <int NC, int EC, bool INDEXED>
__device__ __forceinline__ SplitPlace split_place(const StageArgs& A) {
    using S = SplitShape<NC, EC>;
    SplitPlace p;
    p.lane = threadIdx.x & 63;
    p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    p.fl = p.lane % S::LF;
    p.unit_in_block = p.wave / S::W;
    p.wave_in_unit = p.wave % S::W;
    const uint32_t u = blockIdx.x * S::UNITS + p.unit_in_block;
    p.head = u % A.n_head;
    p.t = u / A.n_head;
    const uint32_t t = min(p.t, A.total_tiles - 1u);   // units past the end load some group and store nothing
    const uint32_t b = t / A.tiles_per_inst, tile = t - b * A.tiles_per_inst;
    const int rl = p.lane / S::LF;
    p.row = p.wave_in_unit * S::ROWS + rl % S::ROWS;
    const uint32_t group = tile * S::GPW + rl / S::ROWS;
    p.exists = p.t < A.total_tiles && group < A.groups;
    p.live = !p.exists ? 0 : INDEXED ? live_rows(A, b, group) : NC;
    p.valid = INDEXED ? p.row < p.live : p.exists;
    const uint32_t g = group < A.groups ? group : 0u;
    const int64_t pos = INDEXED ? slot_position(A, g, p.row) : (int64_t)stage_block(A, g, p.row) * NC + p.row;
    p.off = (int64_t)b * A.N * A.E + pos * A.E + (int64_t)p.head * EC + p.fl * S::F;
    return p;
}

// The pivot row's fragment.  W == 1: through the wave's own slots, in issue order, no barrier.  W > 1: row j of every unit of
// the workgroup goes to `slots` (one of two buffers in turns); the caller's barrier comes between publish and collect.
template <int NC, int EC>
__device__ __forceinline__ void split_publish(const SplitPlace& p, int j, const float (&v)[4], float4* slots) {
    using S = SplitShape<NC, EC>;
    if constexpr (S::W == 1) slots[p.wave * 64 + p.lane] = make_float4(v[0], v[1], v[2], v[3]);
    else if (p.row == j) slots[p.unit_in_block * S::SLOT4 + p.fl] = make_float4(v[0], v[1], v[2], v[3]);
}
template <int NC, int EC>
__device__ __forceinline__ void split_collect(const SplitPlace& p, int j, float (&v)[4], const float4* slots) {
    using S = SplitShape<NC, EC>;
    float4 q;
    if constexpr (S::W == 1) q = slots[p.wave * 64 + ((p.lane & ~((NC - 1) * S::LF)) | (j * S::LF))];
    else q = slots[p.unit_in_block * S::SLOT4 + p.fl];
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}

// forward, and with INVERSE a stage undone; formulas and scaled state of forward_core and inverse_core
template <int NC, int EC, bool INVERSE, bool INDEXED>
__global__ void __launch_bounds__((64 * SplitShape<NC, EC>::NW)) split_forward_kernel(const StageArgs A) {
    using S = SplitShape<NC, EC>;
    constexpr int F = S::F;
    __shared__ float4 slots[2][S::W == 1 ? S::NW * 64 : S::UNITS * S::SLOT4];
    const SplitPlace p = split_place<NC, EC, INDEXED>(A);
    float x[F], a[F], wi[F], wj[F];
    load_frag<F>(A.in0, A.in_dtype, p.off, true, x, A.plane);
    load_frag<F>(A.in1, A.in_dtype, p.off, true, a, A.plane);
    load_w<F>(A, p.head, EC, p.fl, wi, wj);
    const StepTable& T = A.tab;
    if (INDEXED && p.exists && !p.valid) {   // a row past the length passes through
        store_frag<F>(A.out0, A.out_dtype, p.off, true, x, A.plane);
        store_frag<F>(A.out1, A.out_dtype, p.off, true, a, A.plane);
        if (A.aux0) {
            store_frag<F>(A.aux0, NCN_F32, p.off, true, x);
            store_frag<F>(A.aux1, NCN_F32, p.off, true, a);
        }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        x[f] *= T.kappa;
        a[f] *= INVERSE ? T.b_scale : T.a_scale;
    }
#pragma unroll 2
    for (int s = 0; s < NC; ++s) {
        const int j = INVERSE ? NC - 1 - s : s;
        const bool on = !INDEXED || j < p.live;   // a group that a length cuts runs the steps of its live rows; its lanes agree
        float own = 0.f;
        if (on) {
            if constexpr (INVERSE) {
#pragma unroll
                for (int f = 0; f < F; ++f) x[f] = fmaf(T.im, x[f], -a[f]);
            }
            split_publish<NC, EC>(p, j, x, slots[s & 1]);
            own = dot_chain<F>(x, wi);
        }
        if constexpr (S::W > 1) __syncthreads();
        if (on) {
            float xj[F];
            split_collect<NC, EC>(p, j, xj, slots[s & 1]);
            const float c = lane_sum<1, S::LF, true>(own + dot_chain<F>(xj, wj));
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const float z = fmaf(c, xj[f], x[f]);
                const float r = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(z) + 1.0f);
                if constexpr (INVERSE) {
                    a[f] = fmaf(T.bk1, r, fmaf(T.im, a[f], T.bk0));
                } else {
                    a[f] = fmaf(T.m2k2, r, fmaf(T.m, a[f], T.k2));
                    x[f] = fmaf(T.m, x[f], a[f]);
                }
            }
        }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        x[f] *= T.inv_kappa;
        a[f] *= INVERSE ? T.inv_b_scale : T.inv_a_scale;
    }
    store_frag<F>(A.out0, A.out_dtype, p.off, p.valid, x, A.plane);
    store_frag<F>(A.out1, A.out_dtype, p.off, p.valid, a, A.plane);
    if (A.aux0) {
        store_frag<F>(A.aux0, NCN_F32, p.off, p.valid, x);
        store_frag<F>(A.aux1, NCN_F32, p.off, p.valid, a);
    }
}

// reversible backward; formulas and scaled state of backward_core
template <int NC, int EC, bool INDEXED>
__global__ void __launch_bounds__((64 * SplitShape<NC, EC>::NW)) split_backward_kernel(const StageArgs A) {
    using S = SplitShape<NC, EC>;
    constexpr int F = S::F;
    __shared__ float4 slots[2][S::W == 1 ? S::NW * 64 : S::UNITS * S::SLOT4];
    __shared__ float4 parts[2][S::W == 1 ? 1 : S::NW * S::SLOT4];   // [wave]: its rows' share of the pivot gradient
    __shared__ float dw_lds[S::W == 1 ? 1 : S::NW * 2 * EC];
    const SplitPlace p = split_place<NC, EC, INDEXED>(A);
    float Y[F], B[F], G[F], P[F], wi[F], wj[F], dwi[F], dwj[F];
    load_frag<F>(A.in0, A.in_dtype, p.off, true, Y, A.plane);
    load_frag<F>(A.in1, A.in_dtype, p.off, true, B, A.plane);
    load_frag<F>(A.g0, A.g_dtype, p.off, true, G);
    load_frag<F>(A.g1, A.g_dtype, p.off, A.g1 != nullptr, P);
    load_w<F>(A, p.head, EC, p.fl, wi, wj);
    const StepTable& T = A.tab;
    if (INDEXED && p.exists && !p.valid) {   // a row past the length passes through
        store_frag<F>(A.out0, A.out_dtype, p.off, true, G);
        store_frag<F>(A.out1, A.out_dtype, p.off, true, P);
        if (A.aux0) {
            store_frag<F>(A.aux0, NCN_F32, p.off, true, Y);
            store_frag<F>(A.aux1, NCN_F32, p.off, true, B);
        }
    }
    // as if the steps that a cut group skips had been done: G, P carry m^-t
    const float isc = INDEXED && p.live != NC ? pow_steps(T.im, NC - p.live) : 1.0f;
#pragma unroll
    for (int f = 0; f < F; ++f) {
        // lanes without a live row of their own must add nothing to the sums
        Y[f] = p.valid ? Y[f] * T.kappa : 0.f;
        B[f] = p.valid ? B[f] * T.b_scale : 0.f;
        G[f] = p.valid ? G[f] : 0.f;
        P[f] = p.valid ? fmaf(T.om, G[f], P[f]) : 0.f;
        if (INDEXED) {
            G[f] *= isc;
            P[f] *= isc;
        }
        dwi[f] = dwj[f] = 0.f;
    }
    // the lanes of row jp add what the waves left in `buf`: G_j += ku sum, then the P that was held back
    auto add_pivot_share = [&](int jp, const float4* buf) {
        if (p.row == jp) {
            float t[F] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < S::W; ++w) {
                const float4 q = buf[(p.unit_in_block * S::W + w) * S::SLOT4 + p.fl];
                t[0] += q.x; t[1] += q.y; t[2] += q.z; t[3] += q.w;
            }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                G[f] = fmaf(T.ku, t[f], G[f]);
                P[f] = fmaf(T.om, G[f], P[f]);
            }
        }
    };
#pragma unroll 2
    for (int s = 0; s < NC; ++s) {
        const int j = NC - 1 - s;
        const bool on = !INDEXED || j < p.live;
        const float krho = T.krho[s];
        float own = 0.f;
        if (on) {
#pragma unroll
            for (int f = 0; f < F; ++f) Y[f] = fmaf(T.im, Y[f], -B[f]);
            split_publish<NC, EC>(p, j, Y, slots[s & 1]);
            own = dot_chain<F>(Y, wi);
        }
        if constexpr (S::W > 1) __syncthreads();
        if (on) {
            float xj[F];
            split_collect<NC, EC>(p, j, xj, slots[s & 1]);
            if constexpr (S::W > 1) {
                if (s > 0 && (!INDEXED || j + 1 < p.live)) add_pivot_share(j + 1, parts[(s - 1) & 1]);
            }
            const float c = lane_sum<1, S::LF, true>(own + dot_chain<F>(xj, wj));
            float U[F], rh = 0.f;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const float z = fmaf(c, xj[f], Y[f]);
                const float r = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(z) + 1.0f);
                B[f] = fmaf(T.bk1, r, fmaf(T.im, B[f], T.bk0));
                U[f] = P[f] * fmaf(-r, r, r);
                rh = fmaf(U[f], xj[f], rh);
            }
            rh = lane_sum<1, S::LF, true>(rh);
            const float rho_w = krho * rh, rho_ku = T.ku * rh;
            float t[F];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                G[f] = fmaf(T.ku, U[f], G[f]);
                G[f] = fmaf(rho_ku, wi[f], G[f]);
                dwi[f] = fmaf(rho_w, Y[f], dwi[f]);
                dwj[f] = fmaf(rho_w, xj[f], dwj[f]);
                t[f] = fmaf(rh, wj[f], c * U[f]);
            }
            lane_sum_n<S::LF, S::LF * S::ROWS, true, F>(t);   // over the group's rows in this wave
            if constexpr (S::W == 1) {
                const float selku = p.row == j ? T.ku : 0.f;
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    G[f] = fmaf(selku, t[f], G[f]);
                    P[f] = fmaf(T.om, G[f], P[f]);
                }
            } else {
                if (p.lane < S::LF) parts[s & 1][p.wave * S::SLOT4 + p.fl] = make_float4(t[0], t[1], t[2], t[3]);
                const float om = p.row == j ? 0.f : T.om;   // row j's waits for its share
#pragma unroll
                for (int f = 0; f < F; ++f) P[f] = fmaf(om, G[f], P[f]);
            }
        }
    }
    if constexpr (S::W > 1) {
        __syncthreads();
        if (!INDEXED || p.live > 0) add_pivot_share(0, parts[(NC - 1) & 1]);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        G[f] *= T.m_pow_n;
        P[f] = fmaf(P[f], T.m_pow_n, -T.om * G[f]);
    }
    store_frag<F>(A.out0, A.out_dtype, p.off, p.valid, G);
    store_frag<F>(A.out1, A.out_dtype, p.off, p.valid, P);
    if (A.aux0) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            Y[f] *= T.inv_kappa;
            B[f] *= T.inv_b_scale;
        }
        store_frag<F>(A.aux0, NCN_F32, p.off, p.valid, Y);
        store_frag<F>(A.aux1, NCN_F32, p.off, p.valid, B);
    }
    // dW: lanes with the same features, then the unit's waves; unit (t, head) owns the head's slice of partial row t
    lane_sum_n<S::LF, 64, true, F>(dwi);
    lane_sum_n<S::LF, 64, true, F>(dwj);
    float* row = A.dw_partials + (int64_t)p.t * (2 * A.E) + (int64_t)p.head * EC;
    if constexpr (S::W == 1) {
        if (p.lane < S::LF && p.t < A.total_tiles) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                row[p.fl * F + f] = dwi[f];
                row[A.E + p.fl * F + f] = dwj[f];
            }
        }
    } else {
        if (p.lane < S::LF) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                dw_lds[p.wave * 2 * EC + p.fl * F + f] = dwi[f];
                dw_lds[p.wave * 2 * EC + EC + p.fl * F + f] = dwj[f];
            }
        }
        __syncthreads();
        if (p.t < A.total_tiles) {
            for (int k = p.wave_in_unit * 64 + p.lane; k < 2 * EC; k += S::W * 64) {
                float sum = 0.f;
#pragma unroll
                for (int w = 0; w < S::W; ++w) sum += dw_lds[(p.unit_in_block * S::W + w) * 2 * EC + k];
                row[k < EC ? k : A.E + k - EC] = sum;
            }
        }
    }
}

}  // namespace ncn
