// mm_scan_bwd_lanes.hip -- gfx950 backward of the MotifMamba low-rank coupled scan, dstate <= 64.
//
// Reference behaviour: the gradients torch autograd takes through selective_scan_full_matrix_cuda
// (mamba_ssm/ops/selective_scan_interface.py:262-350), the path selective_scan_fn takes for P/Q
// calls with z (selective_scan_interface.py:243-258, the Motif module always passes z), i.e. the
// exact gradients of
//
//     h_t = a_t * h_{t-1} + dt'_t P (Q h_{t-1}) + dt'_t u_t B_t,   a_t = exp(dt'_t A),
//     y_t = C_t . h_t,   out_t = y_t + D u_t,   out_z_t = out_t * silu(z_t).
//
// With g_t = dout_t * silu(z_t) and the state adjoint lam_t = dL / dh_t (a reverse recurrence
// through the transposed transition matrix M_{t+1} = diag(a_{t+1}) + dt'_{t+1} P Q):
//
//     lam_t  = C_t g_t + a_{t+1} * lam_{t+1} + dt'_{t+1} Q^T (P^T lam_{t+1}),     lam_{L-1} = C g
//     dt'_t  = sum_n lam_t (A a_t h_{t-1} + (P q_t) + u_t B_t),    q_t = Q h_{t-1}
//     du_t   = D g_t + dt'_t sum_n lam_t B_t
//     dA    += lam_t dt'_t a_t h_{t-1};  dP += dt'_t lam_t q_t^T;  dQ += dt'_t (P^T lam_t) h_{t-1}^T
//     dB_t  += lam_t dt'_t u_t;  dC_t += g_t h_t;  dD += g_t u_t;  dz, ddelta_bias as the diagonal case.
//
// The design is this file's own. A workgroup owns 16 channels of one (batch, group); the LPR
// consecutive lanes of a channel hold S states each (NP = LPR S: 8 x 2 for dstate <= 16, 16 x 2 for
// <= 32, 16 x 4 for <= 64), so that the sums over a channel's states that feed the recurrences (Q h
// and P^T lam) stay inside 16 lanes: one transposed DPP butterfly each (lane_sums, mm_common.h).
//
//   * The kernel is bound mostly by VALU issue (82 to 90 % of a SIMD's cycles with a coupling, 77 % at
//     dstate 64 without one, at two waves per SIMD, all that the registers of its tile allow; the rest
//     is latency), so what a step costs is its instruction count. The states and (S = 2, rank <= 4) decays
//     of a 16-step tile stay in registers between the recompute and the reverse walk; the P q term
//     of dt' is taken as sum_r q_r (P^T lam)_r from the lane's partials and the u B term as
//     u_t sum_n lam B by the step's owner, so neither costs a multiply per state.
//   * The per-lane sums of du and ddelta and the dB / dC terms go through LDS once per kH steps as
//     (lam B, dt') and (dB, dC) pairs -- one 8-byte access where two 4-byte ones, and DPP
//     butterflies for the sums, took more instructions -- and every lane then finishes one (channel,
//     step) and one (step, state) of them. The row strides of both keep writes and 16-byte reads at
//     the LDS's full rate.
//     Without a coupling (rank 0), and at rank 2 above dstate 16, the dB / dC terms are instead summed
//     over the wave's channels in registers, by swaps of lane halves and of 16-lane rows that reduce two
//     states of both tensors at once, and only the waves' sums go through LDS: a third less LDS (23 KB at
//     dstate 16) and no 16-term sum per row, so three waves per SIMD at rank 0 (8 x 1,536 channels, L
//     1,024, bf16: 1.63 -> 1.14 ms at dstate 64, 8 x 1,024: 0.43 -> 0.36 ms at dstate 32; training steps
//     at rank 2, 4 x 4,096, L 1,024: 1.52 -> 1.33 ms at dstate 32, fp32 3.00 -> 2.38 ms at 64). With 8
//     lanes per channel and a coupling it loses 1% (a third swap stage, two waves per SIMD either way).
//   * Activations and B / C move one element at a time (uniform row bases, fixed 32-bit
//     lane offsets), loaded one tile ahead: any length and row alignment, at
//     about one load per step and lane group.
//   * dB / dC are written as the block's partials and reduced in block order (scan_bwd_reduce_bc);
//     dA, dP, dQ, dD and ddelta_bias take float32 atomics once per lane at the end.
//   * The states at every 16-step tile start come from the forward (its tile_states, dstate <= 16)
//     or from a first pass that recomputes the forward into the caller's workspace.
//
// LDS at rank 2: 40 KB (dstate 16), 39 KB (32), 51 KB (64): two waves per SIMD each; 188 registers at
// dstate 16. 85 VALU instructions per wave-step of 8 channels x 16 states, 114 of 4 x 32. Rank 4 above
// dstate 32 spills 32 to 37 registers, the other instances at most one.
//
// Measured (rank 2, per-channel P/Q), training step of forward and backward: batch 4, 4,096 channels,
// L 2,048, dstate 16, fp16: 1.55 -> 1.26 ms (backward 1.19 -> 0.92) against a kernel with the tile's
// states in LDS, DPP butterflies for the du / ddelta sums and 124 VALU per wave-step; batch 8, 1,024
// channels, L 1,024, dstate 32, bf16: 4.39 -> 0.78 ms against one lane per state.
//
// Compiled once per input type (mm_scan_bwd_lanes_{f16,bf16}.hip include this file).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "mm_common.h"
#include "mm_internal.h"

#ifndef MM_BWD_LANES_TYPE
#define MM_BWD_LANES_TYPE float
#define MM_BWD_LANES_COMMON
#endif

namespace mm {
namespace bwdl {

constexpr int kCh = 16;          // channels per workgroup
constexpr int kT = 16;           // steps per tile
constexpr int kXS = kT + 1;      // sX row stride (float4)
constexpr int kRS = kCh + 2;     // sRed row stride (float2)

template <int LPR, int S, int R>
struct Layout {
    static constexpr bool SW = R == 0 || (R == 2 && LPR == 16);   // dB / dC summed over a wave's channels by lane swaps
    static constexpr int NP = LPR * S;
    static constexpr int NT = kCh * LPR;          // lanes per workgroup
    static constexpr int E = kT / LPR;            // steps per lane of a tile's per-element work
    static constexpr int H = S == 2 || SW ? 8 : 4;   // steps per reduction
    static constexpr int NW = LPR / 4;            // waves
    static constexpr int SR = 32 * S + 4;         // sSum stride of a step (floats)
    static constexpr int BCS = 2 * NP + 4;        // sBC row stride (floats): (B, C) pairs of a step
    static constexpr int RN = H * kRS + 2;        // sRed stride of a state (float2): its H step rows
    static constexpr int PL = LPR + 2;            // sPart stride of a step (float2)
    static constexpr int PC = H * PL + (LPR == 8 ? 8 : 0);   // sPart stride of a channel (float2)
    static constexpr int TPP = NT / (kCh * H);    // lanes that finish one (channel, step)
    static_assert((SW || H * NP == NT) && TPP >= 1, "one dB / dC row per lane");
};

// a + its lane's counterpart in the other half (the other 16-lane row of a pair), b likewise: after the
// swap one add leaves a's sums in the lower half (even rows) and b's in the upper (odd).
__device__ __forceinline__ float swap_add32(float a, float b) {
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b) {
    const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

template <typename T, int LPR, int S, int R>
__global__ void __launch_bounds__(kCh * LPR) __attribute__((amdgpu_waves_per_eu(R == 0 && S == 2 ? 3 : 2)))
scan_bwd_lanes(const mm_scan_bwd_params p, const int64_t ratio, float *const ck, const int64_t ck_batch,
               float *const partB, float *const partC) {
    using Y = Layout<LPR, S, R>;
    constexpr bool SW = Y::SW;
    constexpr int E = Y::E, H = Y::H, BCS = Y::BCS, NP = Y::NP, TPP = Y::TPP;
    constexpr bool AREG = S == 2 && R <= 4;   // the tile's decays stay in registers (else they spill)
    constexpr int RR = R > 0 ? R : 1;    // R = 0: no coupling, the diagonal scan
    constexpr uint32_t SZ = sizeof(T);
    static_assert(R <= LPR, "one transposed reduction per sum set");
    __shared__ __align__(16) float4 sX[kCh * kXS];         // [c][t]: (dt', dt'u, u, g)
    __shared__ __align__(16) float sRaw[kCh * kXS];        // [c][t]: delta + bias
    __shared__ __align__(16) float sBC[kT * BCS];          // [t][n]: (B, C)
    // dB, dC terms: [n][t % H][c] pairs, or (SW) [wave][t % H][lane] sums over the wave's channels.
    __shared__ __align__(16) float2 sRed[SW ? Y::NW * H * Y::SR / 2 : NP * Y::RN];
    float *const sSum = reinterpret_cast<float *>(sRed);
    __shared__ __align__(16) float2 sPart[kCh * Y::PC];    // [c][t % H][k]: lam B and dt' sums of a lane
    __shared__ __align__(16) float sQ[R > 0 ? kT * kCh * R : 4];   // [t][c][r]: Q h_{t-1}

    const int tid = threadIdx.x;
    const int cw = tid / LPR;              // channel of the block
    const int k = tid % LPR;               // states k S .. k S + S - 1
    const int64_t b = blockIdx.y;
    const int64_t d0 = int64_t(blockIdx.x) * kCh;
    const int64_t d = d0 + cw;
    const int64_t g = d0 / ratio;
    const int64_t blk = (d0 - g * ratio) / kCh;
    const int64_t L = p.seqlen;
    const int N = int(p.dstate);
    const int rank = int(p.pq_rank);
    const int64_t n_tiles = (L + kT - 1) / kT;
    const int es = E * k;                  // first step (within a tile) of this lane's elements
    const bool has_z = p.z != nullptr, has_oz = has_z && p.out_z != nullptr;
    const bool softplus = p.delta_softplus != 0;

    // Rows of the block's channels: uniform bases (channel d0), byte offsets of this lane's channel.
    auto in_rows = [&](const void *t, int64_t bs, int64_t ds) {
        return t ? reinterpret_cast<const char *>(reinterpret_cast<const T *>(t) + b * bs + d0 * ds) : nullptr;
    };
    auto out_rows = [&](void *t, int64_t bs, int64_t ds) {
        return t ? reinterpret_cast<char *>(reinterpret_cast<T *>(t) + b * bs + d0 * ds) : nullptr;
    };
    const char *const u_p = in_rows(p.u, p.u_batch_stride, p.u_d_stride);
    const char *const d_p = in_rows(p.delta, p.delta_batch_stride, p.delta_d_stride);
    const char *const go_p = in_rows(p.dout, p.dout_batch_stride, p.dout_d_stride);
    // Without z its loads (and the pre-gate output's) read dout instead: no branch around them.
    const char *const z_p = has_z ? in_rows(p.z, p.z_batch_stride, p.z_d_stride) : go_p;
    const char *const o_p = has_z ? in_rows(p.out, p.out_batch_stride, p.out_d_stride) : go_p;
    char *const du_p = out_rows(p.du, p.du_batch_stride, p.du_d_stride);
    char *const dd_p = out_rows(p.ddelta, p.ddelta_batch_stride, p.ddelta_d_stride);
    char *const dz_p = out_rows(has_z ? p.dz : nullptr, p.dz_batch_stride, p.dz_d_stride);
    char *const oz_p = out_rows(has_oz ? p.out_z : nullptr, p.out_z_batch_stride, p.out_z_d_stride);
    const char *const B_p =
        reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.B) + b * p.B_batch_stride + g * p.B_group_stride);
    const char *const C_p =
        reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.C) + b * p.C_batch_stride + g * p.C_group_stride);
    auto row_off = [&](int c, int64_t ds) { return uint32_t(c * ds) * SZ; };
    // The lane's channel again, opaque: the row offsets below are formed once per tile from it instead of
    // being kept in a register each.
    auto fresh_cw = [&]() {
        int c = cw;
        asm volatile("" : "+v"(c));
        return c;
    };

    // The lane's rows of Q and columns of P in lane_sums order: position t holds rank t ^ ro. Every
    // rank-indexed quantity of the lane (q, P^T lam, dP, dQ) is kept in that order. At dstate <= 16
    // the forward's 8-lane layout forms Q h the same way, so pass 1 reproduces its tile states bit
    // for bit.
    int ro = 0;
    if constexpr (R > 0) ro = lane_rank_offset<LPR, R>(k);
    float An[S], A2[S], Pr[S][RR], Qr[RR][S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int n = k * S + s;
        const bool on = n < N;
        An[s] = on ? p.A[d * p.A_d_stride + n * p.A_dstate_stride] : 0.f;
        A2[s] = An[s] * kLog2e;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const int r = t ^ ro;
            const bool use = on && r < rank;
            Pr[s][t] = use ? p.P[d * p.P_d_stride + n * p.P_dstate_stride + r * p.P_r_stride] : 0.f;
            Qr[t][s] = use ? p.Q[d * p.Q_d_stride + r * p.Q_r_stride + n * p.Q_dstate_stride] : 0.f;
        }
    }
    // Q h over the channel's states, rank t ^ ro in q[t].
    auto qh = [&](const float *h, float (&q)[RR]) {
#pragma unroll
        for (int t = 0; t < R; ++t) {
            q[t] = Qr[t][0] * h[0];
#pragma unroll
            for (int s = 1; s < S; ++s) q[t] = __builtin_fmaf(Qr[t][s], h[s], q[t]);
        }
        if constexpr (R > 0) lane_sums<LPR, R>(q);
    };
    // One step of the recurrence from dt', dt'u, the lane's B and the unscaled q.
    auto step = [&](float dt, float dtu, const float *Bv, const float *a, const float (&qv)[RR], float *h) {
        float q[RR];
#pragma unroll
        for (int r = 0; r < R; ++r) q[r] = qv[r] * dt;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            float w = dtu * Bv[s];
#pragma unroll
            for (int r = 0; r < R; ++r) w = __builtin_fmaf(Pr[s][r], q[r], w);
            h[s] = __builtin_fmaf(a[s], h[s], w);
        }
    };
    const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;

    // Checkpoints [tile][batch][dim][NP] (states past dstate stay 0).
    const int64_t ck_tile = ck_batch * p.dim * NP;
    float *const ckp = ck + (b * p.dim + d) * NP + k * S;

    // B / C staging of a tile: lane (tid / 16, tid % 16) moves step tid % 16 of states tid / 16 + LPR i.
    const int st_t = tid % kT, st_n = tid / kT;
    uint32_t bo[S], co[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {
        const int n = st_n + LPR * i;
        bo[i] = uint32_t((n < N ? n : 0) * p.B_dstate_stride) * SZ;
        co[i] = uint32_t((n < N ? n : 0) * p.C_dstate_stride) * SZ;
    }

    // A tile's global inputs as raw elements, loaded one tile ahead of their use. A row's last, partial
    // tile is right-aligned: position i holds step i - sh of the tile, the sh positions before its first
    // step (clamped to that step) are padding with dt' = u = g = 0 and B = C = 0. Padding in front only
    // meets the tile's entry state and passes it, and the adjoint, on unchanged; behind the last step it
    // would meet that step's own state, where 0 times an infinite state is NaN in dA, dP and dQ.
    struct TileIn {
        uint32_t d[E], u[E], go[E], z[E], o[E], b[S], c[S];
        float hck[S];
    };
    auto padding = [&](int64_t t0) { return int(L - t0 < kT ? kT - (L - t0) : 0); };
    auto fetch = [&](int64_t j, auto full_c, bool with_ck) __attribute__((always_inline)) {
        constexpr bool full = decltype(full_c)::value;
        TileIn r = {};
        const int64_t t0 = j * kT;
        const int c = fresh_cw();
        const uint32_t fo_u = row_off(c, p.u_d_stride), fo_d = row_off(c, p.delta_d_stride);
        const uint32_t fo_go = row_off(c, p.dout_d_stride), fo_z = has_z ? row_off(c, p.z_d_stride) : fo_go;
        const uint32_t fo_o = has_z ? row_off(c, p.out_d_stride) : fo_go;
        const int sh = padding(t0);
        const int64_t so = t0 * SZ;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t eo = uint32_t(max(es - sh + i, 0)) * SZ;
            r.d[i] = load_elem<T>(d_p + so, fo_d + eo);
            r.u[i] = load_elem<T>(u_p + so, fo_u + eo);
            if constexpr (full) {
                r.go[i] = load_elem<T>(go_p + so, fo_go + eo);
                r.z[i] = load_elem<T>(z_p + so, fo_z + eo);
                r.o[i] = load_elem<T>(o_p + so, fo_o + eo);
            }
        }
        const uint32_t to = uint32_t(max(st_t - sh, 0)) * SZ;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            r.b[i] = load_elem<T>(B_p + so, bo[i] + to);
            if constexpr (full) r.c[i] = load_elem<T>(C_p + so, co[i] + to);
        }
        if (with_ck) {
#pragma unroll
            for (int s = 0; s < S; ++s) r.hck[s] = ckp[j * ck_tile + s];
        }
        return r;
    };
    // Tile j's per-step values into LDS (with C when `full`); dz and out_z written.
    auto commit = [&](int64_t j, auto full_c, const TileIn &r) __attribute__((always_inline)) {
        constexpr bool full = decltype(full_c)::value;
        const int64_t t0 = j * kT;
        const int sh = padding(t0);
        const int64_t so = t0 * SZ;
        const int c = fresh_cw();
        const uint32_t fo_dz = row_off(c, p.dz_d_stride), fo_oz = row_off(c, p.out_z_d_stride);
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const bool ev = es - sh + i >= 0;
            const float uu = ev ? elem_f32<T>(r.u[i]) : 0.f;
            float go = 0.f;
            if constexpr (full) {
                go = elem_f32<T>(r.go[i]);
                if (has_z) {
                    const float zz = elem_f32<T>(r.z[i]);
                    const float oo = elem_f32<T>(r.o[i]);
                    const float sg = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-zz * kLog2e));
                    if (ev) {
                        const uint32_t eo = uint32_t(es - sh + i) * SZ;
                        store_elem<T>(dz_p + so, fo_dz + eo, go * oo * sg * (1.f + zz * (1.f - sg)));
                        if (has_oz) store_elem<T>(oz_p + so, fo_oz + eo, oo * zz * sg);
                    }
                    go *= zz * sg;
                }
            }
            const float raw = elem_f32<T>(r.d[i]) + bias;
            const float dt = ev ? (softplus ? softplus_fast(raw) : raw) : 0.f;
            sX[cw * kXS + es + i] = make_float4(dt, dt * uu, uu, ev ? go : 0.f);
            if constexpr (full) sRaw[cw * kXS + es + i] = raw;
        }
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const int n = st_n + LPR * i;
            const bool on = n < N && st_t >= sh;
            const float bv = on ? elem_f32<T>(r.b[i]) : 0.f;
            if constexpr (full)
                *reinterpret_cast<float2 *>(&sBC[st_t * BCS + 2 * n]) = make_float2(bv, on ? elem_f32<T>(r.c[i]) : 0.f);
            else
                sBC[st_t * BCS + 2 * n] = bv;
        }
    };
    constexpr std::true_type kFull{};
    constexpr std::false_type kStates{};

    // ---- Pass 1: the states before every tile (skipped when the forward wrote them) ----
    if (!p.tile_states) {
        float h[S];
#pragma unroll
        for (int s = 0; s < S; ++s) h[s] = 0.f;
        TileIn in = fetch(0, kStates, false);
        for (int64_t j = 0; j < n_tiles; ++j) {
#pragma unroll
            for (int s = 0; s < S; ++s) ckp[j * ck_tile + s] = h[s];
            commit(j, kStates, in);
            if (j + 1 < n_tiles) in = fetch(j + 1, kStates, false);   // in flight during this tile
            __syncthreads();
#pragma unroll
            for (int t = 0; t < kT; ++t) {
                const float2 x = *reinterpret_cast<const float2 *>(&sX[cw * kXS + t]);
                float Bv[S], a[S], q[RR];
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    Bv[s] = sBC[t * BCS + 2 * (k * S + s)];
                    a[s] = decay_exp2(x.x, A2[s]);
                }
                qh(h, q);
                step(x.x, x.y, Bv, a, q, h);
            }
            __syncthreads();
        }
    }

    // ---- Pass 2: tiles in reverse order ----
    float carry[S], dA[S], dP[S][RR], dQ[RR][S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        carry[s] = 0.f;
        dA[s] = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            dP[s][r] = 0.f;
            dQ[r][s] = 0.f;
        }
    }
    // What this lane finishes after every H steps: row (state rd_n, step rd_t) of dB / dC, and the
    // sums of (channel fc, step ft), shared by TPP neighbouring lanes.
    const int rd_t = tid % H, rd_n = tid / H;
    const int fsub = tid % TPP, ft = tid / TPP % H, fc = tid / TPP / H;
    const float Dv = p.D ? p.D[d0 + fc] : 0.f;
    const uint32_t fo_du = row_off(fc, p.du_d_stride), fo_dd = row_off(fc, p.ddelta_d_stride);
    const int64_t Lp = (L + 3) & ~int64_t(3);
    const int64_t slab = ((blk * p.batch + b) * p.n_groups + g) * NP * Lp;
    float *const pB = partB + slab, *const pC = partC + slab;
    const uint32_t rd_off = uint32_t(rd_n) * uint32_t(Lp);
    float dD_acc = 0.f, dbias_acc = 0.f;

    TileIn in = fetch(n_tiles - 1, kFull, true);
    for (int64_t j = n_tiles - 1; j >= 0; --j) {
        const int64_t t0 = j * kT;
        const int sh = padding(t0);
        float hck[S];
#pragma unroll
        for (int s = 0; s < S; ++s) hck[s] = in.hck[s];
        commit(j, kFull, in);
        if (j > 0) in = fetch(j - 1, kFull, true);                  // in flight during this tile
        __syncthreads();
        // Recompute the tile's states from its checkpoint. The LDS reads of a pair of steps are issued
        // before the pair ahead of it is computed.
        float hs[kT][S], as[AREG ? kT : 1][S];
        {
            float h[S], Bn[2][S];
            float2 xn[2];
            auto read = [&](int t) __attribute__((always_inline)) {
                xn[t & 1] = *reinterpret_cast<const float2 *>(&sX[cw * kXS + t]);
#pragma unroll
                for (int s = 0; s < S; ++s) Bn[t & 1][s] = sBC[t * BCS + 2 * (k * S + s)];
            };
            read(0);
            read(1);
#pragma unroll
            for (int s = 0; s < S; ++s) h[s] = hck[s];
            static_for<0, kT / 2>([&](auto pair_c) __attribute__((always_inline)) {
                constexpr int t0p = 2 * decltype(pair_c)::value;
                float2 x2[2] = {xn[0], xn[1]};
                float B2[2][S];
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    B2[0][s] = Bn[0][s];
                    B2[1][s] = Bn[1][s];
                }
                if constexpr (t0p + 2 < kT) {
                    read(t0p + 2);
                    read(t0p + 3);
                }
                static_for<0, 2>([&](auto i_c) __attribute__((always_inline)) {
                    constexpr int t = t0p + decltype(i_c)::value;
                    const float2 x = x2[t & 1];
                    float a[S], q[RR];
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        a[s] = decay_exp2(x.x, A2[s]);
                        if constexpr (AREG) as[t][s] = a[s];
                    }
                    qh(h, q);
                    if constexpr (R > 0) {
                        if (k == 0) {   // rank order: lane 0 of the channel has rank offset 0
#pragma unroll
                            for (int r = 0; r < R; r += 2)
                                *reinterpret_cast<float2 *>(&sQ[(t * kCh + cw) * R + r]) = make_float2(q[r], q[r + 1]);
                        }
                    }
                    step(x.x, x.y, B2[t & 1], a, q, h);
#pragma unroll
                    for (int s = 0; s < S; ++s) hs[t][s] = h[s];
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        // sQ is written by one lane of a channel and read by the others, all lanes of one wave, whose LDS
        // accesses the hardware keeps in order. The fences keep the compiler from moving a read before
        // the store (the wave barrier alone orders no memory); at this scope they emit no instruction.
        if constexpr (R > 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        }
        float4 xn[2];
        float Bn[2][S], Cn[2][S], qn[2][RR];
        auto read = [&](int t) __attribute__((always_inline)) {
            xn[t & 1] = sX[cw * kXS + t];                    // dt', dt'u, u, g
#pragma unroll
            for (int s = 0; s < S; s += 2) {
                const float4 v = *reinterpret_cast<const float4 *>(&sBC[t * BCS + 2 * (k * S + s)]);
                Bn[t & 1][s] = v.x; Cn[t & 1][s] = v.y; Bn[t & 1][s + 1] = v.z; Cn[t & 1][s + 1] = v.w;
            }
            if constexpr (R == 2) {
                const float2 v = *reinterpret_cast<const float2 *>(&sQ[(t * kCh + cw) * R]);
                qn[t & 1][0] = ro ? v.y : v.x;
                qn[t & 1][1] = ro ? v.x : v.y;
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) qn[t & 1][r] = sQ[(t * kCh + cw) * R + (r ^ ro)];
            }
        };
        read(kT - 1);
        read(kT - 2);
        float4 x2[2];
        float B2[2][S], C2[2][S], q2[2][RR];
        static_for<0, kT / H>([&](auto part_c) __attribute__((always_inline)) {
            constexpr int tg = kT - H - H * decltype(part_c)::value;   // first step of this part
            static_for<0, H>([&](auto step_c) __attribute__((always_inline)) {
                constexpr int ti = H - 1 - decltype(step_c)::value, t = tg + ti;
                if constexpr (t & 1) {                     // the first of a pair: its reads, then the next pair's
                    x2[0] = xn[0];
                    x2[1] = xn[1];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
#pragma unroll
                        for (int s = 0; s < S; ++s) {
                            B2[i][s] = Bn[i][s];
                            C2[i][s] = Cn[i][s];
                        }
#pragma unroll
                        for (int r = 0; r < R; ++r) q2[i][r] = qn[i][r];
                    }
                    if constexpr (t >= 3) {
                        read(t - 2);
                        read(t - 3);
                    }
                }
                const float4 x = x2[t & 1];
                const float *const Bv = B2[t & 1], *const Cv = C2[t & 1];
                float lam[S], sv[RR], q[RR], tb[S], tc[S];
#pragma unroll
                for (int s = 0; s < S; ++s) lam[s] = __builtin_fmaf(Cv[s], x.w, carry[s]);
                // P^T lam over the channel's states, rank t ^ ro at position t (as Pr, Qr, dP, dQ),
                // and the lane's part of sum_n lam P q = sum_r q_r (P^T lam)_r.
                float pdd = 0.f, pgb = 0.f;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    q[r] = q2[t & 1][r];
                    sv[r] = Pr[0][r] * lam[0];
#pragma unroll
                    for (int s = 1; s < S; ++s) sv[r] = __builtin_fmaf(Pr[s][r], lam[s], sv[r]);
                    pdd = __builtin_fmaf(q[r], sv[r], pdd);
                }
                if constexpr (R > 0) lane_sums<LPR, R>(sv);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    sv[r] *= x.x;
                    q[r] *= x.x;
                }
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    float a, hp;
                    if constexpr (AREG) a = as[t][s];
                    else a = decay_exp2(x.x, A2[s]);
                    if constexpr (t > 0) hp = hs[t - 1][s];
                    else hp = hck[s];
                    const float w = lam[s] * (a * hp);
                    dA[s] = __builtin_fmaf(x.x, w, dA[s]);
                    pdd = __builtin_fmaf(An[s], w, pdd);
                    pgb = __builtin_fmaf(lam[s], Bv[s], pgb);
                    float c = a * lam[s];                            // into step t - 1
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        dP[s][r] = __builtin_fmaf(lam[s], q[r], dP[s][r]);
                        dQ[r][s] = __builtin_fmaf(sv[r], hp, dQ[r][s]);
                        c = __builtin_fmaf(Qr[r][s], sv[r], c);
                    }
                    carry[s] = c;
                    if constexpr (SW) {
                        tb[s] = lam[s] * x.y;
                        tc[s] = x.w * hs[t][s];
                    } else {
                        sRed[(k * S + s) * Y::RN + ti * kRS + cw] = make_float2(lam[s] * x.y, x.w * hs[t][s]);
                    }
                }
                if constexpr (SW) {
                    // Sums over the wave's 64 / LPR channels (lane / LPR): the swap of lane halves adds
                    // dB in the lower and dC in the upper one, the swap of 16-lane rows then state 2 i in
                    // the even and 2 i + 1 in the odd rows; with 8 lanes per channel a row holds two.
#pragma unroll
                    for (int i = 0; i < S; i += 2) {
                        const float a = swap_add32(tb[i], tc[i]), b2 = swap_add32(tb[i + 1], tc[i + 1]);
                        float v = swap_add16(a, b2);
                        if constexpr (LPR == 8) v = dpp_add<0x128>(v);      // row_ror:8
                        sSum[((tid >> 6) * H + ti) * Y::SR + 32 * i + (tid & 63)] = v;
                    }
                }
                sPart[cw * Y::PC + ti * Y::PL + k] = make_float2(pgb, pdd);
                if constexpr (t % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            });
            // The accumulators are complete here: without this the compiler sinks their updates past
            // the reductions below and keeps the operands of every step alive until there.
#pragma unroll
            for (int s = 0; s < S; ++s) {
                asm volatile("" : "+v"(dA[s]));
#pragma unroll
                for (int r = 0; r < R; ++r) asm volatile("" : "+v"(dP[s][r]), "+v"(dQ[r][s]));
            }
            __syncthreads();
            if constexpr (SW) {   // dB / dC of S (step, state)s: the waves' sums added in order.
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    const int e = tid + Y::NT * i, rt = e % H, q = e / H, tz = q / NP, n = q % NP;
                    const int at = 32 * ((n % S) & ~1) + (tz * 2 + (n & 1)) * 16 + n / S;
                    float acc = sSum[rt * Y::SR + at];
#pragma unroll
                    for (int w = 1; w < Y::NW; ++w) acc += sSum[(w * H + rt) * Y::SR + at];
                    if (tg + rt - sh >= 0 && n < N)
                        (tz == 0 ? pB : pC)[uint32_t(n) * uint32_t(Lp) + uint32_t(t0) + uint32_t(tg + rt - sh)] = acc;
                }
            } else {   // dB / dC of one (step, state) over the block's 16 channels, added pairwise in a fixed order.
                const float4 *rv = reinterpret_cast<const float4 *>(&sRed[rd_n * Y::RN + rd_t * kRS]);
                float vb[kCh / 2], vc[kCh / 2];
#pragma unroll
                for (int i = 0; i < kCh / 2; ++i) {
                    const float4 v = rv[i];
                    vb[i] = v.x + v.z;
                    vc[i] = v.y + v.w;
                }
#pragma unroll
                for (int w = 1; w < kCh / 2; w *= 2) {
#pragma unroll
                    for (int i = 0; i < kCh / 2; i += 2 * w) {
                        vb[i] += vb[i + w];
                        vc[i] += vc[i + w];
                    }
                }
                if (rd_t - sh + tg >= 0 && rd_n < N) {
                    const uint32_t o = rd_off + uint32_t(t0) + uint32_t(rd_t - sh + tg);
                    pB[o] = vb[0];
                    pC[o] = vc[0];
                }
            }
            {   // du / ddelta of one (channel, step).
                const int t = tg + ft;
                const float4 *pv = reinterpret_cast<const float4 *>(
                    &sPart[fc * Y::PC + ft * Y::PL + fsub * (LPR / TPP)]);
                float gb = 0.f, dd = 0.f;
#pragma unroll
                for (int i = 0; i < LPR / TPP / 2; ++i) {
                    const float4 v = pv[i];
                    gb += v.x + v.z;
                    dd += v.y + v.w;
                }
                if constexpr (TPP >= 2) {
                    gb = dpp_add<0xB1>(gb);                          // quad_perm [1,0,3,2]
                    dd = dpp_add<0xB1>(dd);
                }
                if constexpr (TPP >= 4) {
                    gb = dpp_add<0x4E>(gb);                          // quad_perm [2,3,0,1]
                    dd = dpp_add<0x4E>(dd);
                }
                const float4 x = sX[fc * kXS + t];
                const float raw = sRaw[fc * kXS + t];
                if (ft - sh + tg >= 0) {
                    const int64_t so = t0 * SZ;
                    const uint32_t to = uint32_t(ft - sh + tg) * SZ;
                    if (fsub == 0) {
                        store_elem<T>(du_p + so, fo_du + to, __builtin_fmaf(Dv, x.w, x.x * gb));
                        dD_acc = __builtin_fmaf(x.w, x.z, dD_acc);
                    }
                    if (fsub == TPP / 2) {
                        dd = __builtin_fmaf(x.z, gb, dd);
                        const float sg = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-raw * kLog2e));
                        if (softplus && raw <= 20.f) dd *= sg;
                        store_elem<T>(dd_p + so, fo_dd + to, dd);
                        dbias_acc += dd;
                    }
                }
            }
            __syncthreads();   // sRed, sPart (and after the tile's last part sX, sBC) are rewritten
        });
    }
    // The strides and pointers below are read from the kernel arguments again: kept from the kernel's
    // start they would spill the scalar registers of the tile loop. dP[s][t] and dQ[t][s] hold rank t ^ ro.
#ifdef __HIP_DEVICE_COMPILE__
    auto *pa = (const __attribute__((address_space(4))) mm_scan_bwd_params *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(pa));
#else
    const mm_scan_bwd_params *pa = &p;
#endif
    const auto &pt = *pa;
    const bool shared_pq = R > 0 && pt.dP_d_stride == 0 && pt.dQ_d_stride == 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int n = k * S + s;
        if (n >= N) continue;
        atomicAdd(pt.dA + d * pt.dA_d_stride + n * pt.dA_dstate_stride, dA[s]);
        if (shared_pq) continue;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const int r = t ^ ro;
            if (r >= rank) continue;
            atomicAdd(pt.dP + d * pt.dP_d_stride + n * pt.dP_dstate_stride + r * pt.dP_r_stride, dP[s][t]);
            atomicAdd(pt.dQ + d * pt.dQ_d_stride + r * pt.dQ_r_stride + n * pt.dQ_dstate_stride, dQ[t][s]);
        }
    }
    if (pt.dD && fsub == 0) atomicAdd(pt.dD + d0 + fc, dD_acc);
    if (pt.ddelta_bias && fsub == TPP / 2) atomicAdd(pt.ddelta_bias + d0 + fc, dbias_acc);
    if constexpr (R > 0) if (shared_pq) {
        // One dP / dQ shared by every channel: the block's 16 channels are summed in LDS first, so
        // that each element takes one atomic per block, not one per lane.
        float *const sum = reinterpret_cast<float *>(sRed);           // [dP | dQ][n][r][c]
        static_assert(2 * NP * R * kCh <= (SW ? Y::NW * H * Y::SR : 2 * NP * Y::RN), "the shared-P/Q sums fit sRed");
        __syncthreads();
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const int r = t ^ ro;
                sum[((0 * NP + k * S + s) * R + r) * kCh + cw] = dP[s][t];
                sum[((1 * NP + k * S + s) * R + r) * kCh + cw] = dQ[t][s];
            }
        }
        __syncthreads();
        for (int e = tid; e < 2 * NP * R; e += Y::NT) {
            const int which = e / (NP * R), n = (e / R) % NP, r = e % R;
            if (n >= N || r >= rank) continue;
            const float4 *v = reinterpret_cast<const float4 *>(&sum[e * kCh]);
            float q4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) q4[i] = (v[i].x + v[i].y) + (v[i].z + v[i].w);
            const float acc = (q4[0] + q4[1]) + (q4[2] + q4[3]);
            if (which == 0) atomicAdd(pt.dP + n * pt.dP_dstate_stride + r * pt.dP_r_stride, acc);
            else atomicAdd(pt.dQ + r * pt.dQ_r_stride + n * pt.dQ_dstate_stride, acc);
        }
    }
}

}  // namespace bwdl

// ------------------------------------------------------------------------------------------------
// Host side.
// ------------------------------------------------------------------------------------------------
#ifdef MM_BWD_LANES_COMMON
bool bwd_lanes_ok(const mm_scan_bwd_params &p) {
    if (!p.is_variable_B || !p.is_variable_C || p.dstate < 1 || p.dstate > 64 || p.seqlen < 1) return false;
    // Rank 8 with four states per lane would hold 128 values of P, Q, dP and dQ in registers alone.
    if (p.P && (p.pq_rank < 1 || p.pq_rank > (p.dstate > 32 ? 4 : 8))) return false;
    if (p.dim % 16 != 0 || (p.dim / p.n_groups) % 16 != 0) return false;
    // 32-bit byte offsets from the block's first channel row and from the (batch, group) of B / C,
    // and element offsets inside one block's slab.
    const int64_t eb = p.itype == MM_FLOAT32 ? 4 : 2, lim = int64_t(1) << 32;
    const int64_t ds[] = {p.u_d_stride, p.delta_d_stride, p.dout_d_stride, p.du_d_stride, p.ddelta_d_stride,
                          p.z ? p.z_d_stride : 0, p.z ? p.out_d_stride : 0, p.z ? p.dz_d_stride : 0,
                          p.z && p.out_z ? p.out_z_d_stride : 0};
    for (int64_t s : ds)
        if (s < 0 || (15 * s + p.seqlen + 16) * eb >= lim) return false;
    for (int64_t s : {p.B_dstate_stride, p.C_dstate_stride})
        if (s < 0 || ((p.dstate - 1) * s + p.seqlen + 16) * eb >= lim) return false;
    const int64_t row = 2 * (p.dim / 16) * bwd_lanes_np(p) * ((p.seqlen + 3) & ~int64_t(3)) * int64_t(sizeof(float));
    // One batch row's slabs may take 4 GiB at dstate > 16 (the general kernel adds with atomics there).
    return 64 * (p.seqlen + 16) < lim && (p.dstate <= 16 || row <= lim);
}

int bwd_lanes_np(const mm_scan_bwd_params &p) { return p.dstate <= 16 ? 16 : p.dstate <= 32 ? 32 : 64; }

// Batch rows per launch: their slabs share at most 4 GiB of workspace.
int64_t bwd_lanes_batch(const mm_scan_bwd_params &p) {
    const int64_t row = 2 * (p.dim / 16) * bwd_lanes_np(p) * ((p.seqlen + 3) & ~int64_t(3)) * int64_t(sizeof(float));
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>((int64_t(1) << 32) / std::max<int64_t>(row, 1), 65535));
    return std::min<int64_t>(p.batch, most);
}
#endif

namespace bwdl {
template <typename T, int LPR, int S, int R>
int launch(const mm_scan_bwd_params &p, hipStream_t s, float *ck, int64_t ck_batch, float *partB, float *partC) {
    hipLaunchKernelGGL((scan_bwd_lanes<T, LPR, S, R>), dim3(unsigned(p.dim / kCh), unsigned(p.batch)),
                       dim3(kCh * LPR), 0, s, p, p.dim / p.n_groups, ck, ck_batch, partB, partC);
    return launch_status("scan_bwd_lanes");
}
}  // namespace bwdl

template <typename T>
int launch_bwd_lanes(const mm_scan_bwd_params &p, hipStream_t s, float *ck, int64_t ck_batch, float *partB,
                     float *partC) {
    const int np = bwd_lanes_np(p);
    if (!p.P) {
        if (np == 16) return bwdl::launch<T, 8, 2, 0>(p, s, ck, ck_batch, partB, partC);
        if (np == 32) return bwdl::launch<T, 16, 2, 0>(p, s, ck, ck_batch, partB, partC);
        return bwdl::launch<T, 16, 4, 0>(p, s, ck, ck_batch, partB, partC);
    }
    if (np == 16) {
        if (p.pq_rank <= 2) return bwdl::launch<T, 8, 2, 2>(p, s, ck, ck_batch, partB, partC);
        if (p.pq_rank <= 4) return bwdl::launch<T, 8, 2, 4>(p, s, ck, ck_batch, partB, partC);
        return bwdl::launch<T, 8, 2, 8>(p, s, ck, ck_batch, partB, partC);
    }
    if (np == 32) {
        if (p.pq_rank <= 2) return bwdl::launch<T, 16, 2, 2>(p, s, ck, ck_batch, partB, partC);
        if (p.pq_rank <= 4) return bwdl::launch<T, 16, 2, 4>(p, s, ck, ck_batch, partB, partC);
        return bwdl::launch<T, 16, 2, 8>(p, s, ck, ck_batch, partB, partC);
    }
    if (p.pq_rank <= 2) return bwdl::launch<T, 16, 4, 2>(p, s, ck, ck_batch, partB, partC);
    return bwdl::launch<T, 16, 4, 4>(p, s, ck, ck_batch, partB, partC);
}

template int launch_bwd_lanes<MM_BWD_LANES_TYPE>(const mm_scan_bwd_params &, hipStream_t, float *, int64_t, float *,
                                                 float *);

}  // namespace mm
