// mm_scan_pq.hip -- gfx950 forward selective scan with the MotifMamba low-rank P/Q coupling.
//
// Reference behaviour: selective_scan_full_matrix_cuda (mamba_ssm/ops/selective_scan_interface.py:
// 262-350), the path selective_scan_fn takes for P/Q (selective_scan_interface.py:237-259), and the
// dense CUDA forward selective_scan_fwd_dense_pq_kernel (csrc/selective_scan/
// selective_scan_fwd_kernel.cuh:159-251, one thread per (batch, channel) row). The recurrence
//
//     h_t = exp(dt'_t A[d,:]) * h_{t-1} + dt'_t P_d (Q_d h_{t-1}) + dt'_t u_t B_t
//
// couples every state of a row to every other one through the rank-R product, so a row is not a
// set of independent per-state scans: each state needs Q h_{t-1} before it can take step t. The
// design of this file is its own:
//
//   scan_fwd_pq_tiled<T, S, LPR, R>   a wave64 owns 64/LPR channels of one (batch, group), at
//       dstate above 32 four of them in a workgroup; the LPR consecutive lanes of a channel hold S
//       states each (S * LPR >= dstate, padded with states whose A, P, Q, B and C are zero, which stay zero). Per step each lane forms its partial
//       Q h over its S states, a DPP butterfly inside the LPR lanes sums the partials (every lane
//       ends with the same bits; where the rank is at most LPR one transposed butterfly serves all
//       R sums, lane_sums in mm_common.h), and the lane updates its S states with
//       P (dt' q) + dt' u B.
//       The lane's rows of P and Q live in registers for the whole sequence. (16-bit inputs with
//       16 lanes of one state and rank <= 2 carry the butterfly's total from step to step and form
//       the next partial as Q (a h + dt' u B) + (Q P) q, which shortens the dependent chain.)
//       * B and C of the (batch, group) are staged per 32-step tile in LDS as float32, [step][state],
//         and each step reads the lane's S states as one vector.
//       * dt' = softplus(delta + bias) and dt' u are computed once per (channel, step): each lane
//         owns 32/LPR consecutive steps of its channel per tile and shares them through LDS.
//       * Per-lane partial sums of y = sum_n C_n h_n go back through LDS; the owner of the step adds
//         the LPR partials in lane order, applies D u and the silu(z) gate and stores.
//       * Global loads for tile i+1 are issued before the scan of tile i.
//   scan_fwd_pq_step<T, LPR, U>   one time step, four states per lane (the Motif decode step).
//   scan_fwd_pq_lanes<T, LPR, R>   four states per lane in registers, any strides and lengths,
//       constant B/C: whatever else the tiled kernel does not take.
//   scan_fwd_pq_rowlane<T>   one lane per row, the row's states in LDS, P/Q read through the cache
//       every step: the same for dstate 65 to 256.
#include <hip/hip_runtime.h>

#include <stdlib.h>

#include <algorithm>

#include <type_traits>

#include "mm_common.h"
#include "mm_internal.h"

// Compiled once per input type (mm_scan_pq_{f16,bf16}.hip include this file).
#ifndef MM_PQ_TYPE
#define MM_PQ_TYPE float
#define MM_PQ_COMMON
#endif

namespace mm {
namespace pq {

constexpr int kT = 32;      // sequence steps per tile
constexpr int kPad = 36;    // LDS row stride (floats) of per-channel step rows: 16-B aligned, spreads banks
constexpr int kMaxRank = 8; // selective_scan.cpp:359

// S consecutive floats of LDS (16-B, 8-B or 4-B aligned by construction).
template <int S>
__device__ __forceinline__ void lds_read_vec(const float *src, float *o) {
    if constexpr (S == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(src);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else if constexpr (S == 2) {
        const float2 v = *reinterpret_cast<const float2 *>(src);
        o[0] = v.x; o[1] = v.y;
    } else {
        o[0] = *src;
    }
}

// Waves per workgroup that share the staged B and C. At dstate above 32 a lane alone would load and stage
// four vectors of each per tile, more than the registers hold beside the scan; four waves take one each
// (16 channels: 8 x 2,048 channels, L 2,048, bf16, dstate 64: 0.77 -> 0.53 ms, with P/Q of rank 2 at batch 4
// 0.71 -> 0.43 ms). At dstate 32 two waves would land on the same SIMDs where the grid fills each once
// (P/Q, 4 x 2,048 channels, L 2,047: 0.28 against 0.43 ms).
constexpr int waves_sharing(int np) { return np > 32 ? 4 : 1; }

template <typename T, int N>
__device__ __forceinline__ void pin_raw(RawVec<T, N> &r) {
#pragma unroll
    for (auto &w : r.w) asm volatile("" : "+v"(w));
}

// R = 0: no coupling, the diagonal scan of the dstate values the dstate-16 kernels do not take, with
// the chunk states in its form, (prod of the decays since step 0, h); otherwise (1, h), the P/Q form.
// 8 x 1,536 channels, L 1,024, bf16, dstate 64: 0.436 -> 0.287 ms against the rank-2 instance with a
// zero pair; 4 x 2,048 channels, L 2,048, dstate 32: 0.28 -> 0.18 ms, dstate 8: 0.20 -> 0.14 ms.
// VEC: every row starts 16-byte aligned and L is a multiple of 8. Without it (any L, any row
// alignment) the same vectors move through global accesses that need only the element's alignment,
// and the last, partial tile moves element by element: 3 x 4,320 channels, L 1,797, dstate 16, rank
// 2, fp16 0.25 ms against 0.45 ms on copies padded to whole tiles.
template <typename T, int S, int LPR, int R, bool VEC = true>
__global__ void __launch_bounds__(64 * waves_sharing(S * LPR)) __attribute__((amdgpu_waves_per_eu(2)))
scan_fwd_pq_tiled(const mm_scan_fwd_params p, const int64_t ratio, const int32_t blocks_per_group) {
    constexpr bool DX = R == 0;
    constexpr int RR = R > 0 ? R : 1;
    constexpr int NP = S * LPR;            // padded states per channel
    constexpr int CPW = 64 / LPR;          // channels per wave
    constexpr int W = waves_sharing(NP);   // waves per workgroup, sharing the staged B and C
    constexpr int NU = NP / 16 / W;        // units of B and C a lane stages per tile
    constexpr int E = kT / LPR;            // prologue / epilogue steps per lane per tile
    // sBC row stride (floats): NP B values, then NP C values. The staging writes, for one element
    // position, lanes (state n = lane / 4, step block q = lane % 4) at q 8 BCS + n: with BCS = 2 NP + 2
    // (S <= 2; the scan reads S-vectors of 8 bytes) 8 BCS = 16 mod 64, so the 64 lanes cover 64
    // consecutive banks; S = 4 needs 16-byte aligned rows (2 NP + 4).
    constexpr int BCS = S <= 2 ? 2 * NP + 2 : 2 * NP + 4;
    static_assert(NU >= 1 && E >= 2 && E % 2 == 0 && 2 * CPW <= 64, "tile shape");
    __shared__ __align__(16) float sBC[kT * BCS];
    // Per wave, during the scan: dt' rows then dt'u rows of its channels; after it: the y partials.
    __shared__ __align__(16) float sX[W * 64 * kPad];
    const int wave = threadIdx.x / 64;
    float *sDt = sX + wave * (64 * kPad);
    float *sDu = sDt + CPW * kPad;
    float *sY = sDt;

    const int lane = threadIdx.x % 64;
    const int cw = lane / LPR;             // channel slot in the wave
    const int k = lane % LPR;              // state slice: states k S .. k S + S - 1
    const int64_t b = blockIdx.y;
    const int64_t g = blockIdx.x / blocks_per_group;
    const int64_t cl = int64_t(blockIdx.x % blocks_per_group) * (CPW * W) + wave * CPW + cw;  // channel within the group
    const bool active = cl < ratio;
    const int64_t d = g * ratio + (active ? cl : ratio - 1);  // inactive slots mirror a real channel
    const int64_t L = p.seqlen;
    const int N = int(p.dstate);
    const int rank = int(p.pq_rank);

    const T *zp = p.z ? reinterpret_cast<const T *>(p.z) + b * p.z_batch_stride + d * p.z_d_stride : nullptr;
    const T *Bg = reinterpret_cast<const T *>(p.B) + b * p.B_batch_stride + g * p.B_group_stride;
    const T *Cg = reinterpret_cast<const T *>(p.C) + b * p.C_batch_stride + g * p.C_group_stride;

    // XK: the carried form described below. TS: the coupling's R sums over the channel's lanes are one transposed
    // reduction (lane_sums, R <= LPR), which wants the lane's rows of Q and columns of P in its
    // order: position t holds rank t ^ ro.
    constexpr bool XK = LPR == 16 && S == 1 && R > 0 && R <= 2 && !std::is_same<T, float>::value;
    constexpr bool TS = R > 0 && R <= LPR && !XK;
    int ro = 0;
    if constexpr (TS) ro = lane_rank_offset<LPR, R>(k);
    float A2[S], h[S], Pr[S][RR], Qr[RR][S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int n = k * S + s;
        const bool on = n < N;
        A2[s] = on ? p.A[d * p.A_d_stride + n * p.A_dstate_stride] * kLog2e : 0.f;
        h[s] = 0.f;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const int j = t ^ ro;
            const bool use = on && j < rank;
            Pr[s][t] = use ? p.P[d * p.P_d_stride + n * p.P_dstate_stride + j * p.P_r_stride] : 0.f;
            Qr[t][s] = use ? p.Q[d * p.Q_d_stride + j * p.Q_r_stride + n * p.Q_dstate_stride] : 0.f;
        }
    }
    // With 16 lanes of one state per channel (dstate <= 16, chosen when their waves fit one per
    // SIMD, where each step's dependent chain sets the time) and rank <= 2, the coupling carries
    // gq = Q h_{t-1} over all states of the channel from step to step (h = 0 before the first
    // step) and forms the next one as Q hb + K q with K = Q P over the lane's states (R x R): the
    // chain from gq to the next gq is then q, R fmas and the butterfly instead of q, the P fmas,
    // the S-term dot product and the butterfly, for R^2 + R S more VALU per step. Measured at one
    // wave per SIMD: -8 % at one state per lane, +4 % at two (the extra VALU outweigh the shorter
    // chain); +10 % at two waves per SIMD with 8 lanes, where issue sets the time. 16-bit inputs
    // only: float32 callers keep the direct Q h, whose rounding the long-sequence float32 checks
    // pin; 16-bit outputs round far above the float32 rounding difference of the two forms.
    float Kr[RR][RR], gq[RR];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        gq[r] = 0.f;
#pragma unroll
        for (int r2 = 0; r2 < R; ++r2) {
            float acc = Qr[r][0] * Pr[0][r2];
#pragma unroll
            for (int s = 1; s < S; ++s) acc = __builtin_fmaf(Qr[r][s], Pr[s][r2], acc);
            Kr[r][r2] = acc;
        }
    }
    const float Dv = p.D ? p.D[d] : 0.f;
    const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
    const bool softplus = p.delta_softplus != 0;
    const int es = E * k;                  // first step (within a tile) of this lane's elements
    const int64_t n_chunks = (L + MM_SCAN_CHUNK - 1) / MM_SCAN_CHUNK;
    float cum_dt = 0.f;                    // R = 0: running sum of dt' (prod a = exp2(A log2e cum_dt))
    // Checkpoints for the backward: the S states of this lane before every 16-step tile.
    const int64_t ck_tile = p.batch * p.dim * 16;
    float *const ckp = (p.tile_states && active) ? p.tile_states + (b * p.dim + d) * 16 + k * S : nullptr;
    auto put_ck = [&](int64_t j) {
#pragma unroll
        for (int s = 0; s < S; ++s) ckp[j * ck_tile + s] = h[s];
    };

    // The loads of u, delta and z go through buffer resources: the rows of the workgroup's channels from
    // its first channel dw, with 32-bit byte offsets per lane (the host checks that every offset of
    // these rows fits). A whole tile adds its start as a scalar offset; only the last, partial
    // tile clamps per lane. (B and C, a tensor per lane, keep per-lane pointers: a resource
    // descriptor must be uniform.)
    constexpr uint32_t SZ = sizeof(T);
    const int64_t dw = g * ratio + int64_t(blockIdx.x % blocks_per_group) * (CPW * W);
    const int64_t dl = d - dw;             // 0 .. CPW W - 1 (inactive slots mirror the group's last channel)
    const __amdgpu_buffer_rsrc_t rs_u = buffer_rsrc(reinterpret_cast<const T *>(p.u) + b * p.u_batch_stride + dw * p.u_d_stride);
    const __amdgpu_buffer_rsrc_t rs_d =
        buffer_rsrc(reinterpret_cast<const T *>(p.delta) + b * p.delta_batch_stride + dw * p.delta_d_stride);
    const __amdgpu_buffer_rsrc_t rs_z =    // (p.z, not zp: the condition must be uniform)
        buffer_rsrc(p.z ? reinterpret_cast<const T *>(p.z) + b * p.z_batch_stride + dw * p.z_d_stride : nullptr);
    const uint32_t fo_u = uint32_t(dl * p.u_d_stride) * SZ, fo_d = uint32_t(dl * p.delta_d_stride) * SZ;
    const uint32_t fo_z = uint32_t(dl * p.z_d_stride) * SZ;
    // The outputs likewise (stores only from lanes of real channels, at existing steps).
    const __amdgpu_buffer_rsrc_t rs_o =
        buffer_rsrc(p.out ? reinterpret_cast<T *>(p.out) + b * p.out_batch_stride + dw * p.out_d_stride : nullptr);
    const __amdgpu_buffer_rsrc_t rs_oz =
        buffer_rsrc(p.out_z ? reinterpret_cast<T *>(p.out_z) + b * p.out_z_batch_stride + dw * p.out_z_d_stride : nullptr);
    const uint32_t fo_o = uint32_t(dl * p.out_d_stride + es) * SZ, fo_oz = uint32_t(dl * p.out_z_d_stride + es) * SZ;

    // B and C of the (batch, group) through buffer resources too. Per 32-step tile every lane stages
    // NU units of each tensor: unit u is the 8 steps 8 (u % 4) .. + 7 of state u / 4, thread t of the
    // 64 W takes units t + 64 W i (4 NP in all): one 8-element load from B and one from C each (a 32-bit
    // offset per lane, the tile start as a scalar offset). Units of padded states (u / 4 >= dstate)
    // and, in a last partial tile, units past L (L is a multiple of 8: a unit is all in or all out)
    // are zeroed once when loaded, so the staging below writes every unit unconditionally.
    const __amdgpu_buffer_rsrc_t rs_B = buffer_rsrc(Bg), rs_C = buffer_rsrc(Cg);
    const int u_n = threadIdx.x / 4, u_q = threadIdx.x % 4;
    bool u_on[NU];
    uint32_t fo_B[NU], fo_C[NU];
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const int n = u_n + 16 * W * i;
        u_on[i] = n < N;
        fo_B[i] = uint32_t((u_on[i] ? n : 0) * p.B_dstate_stride) * SZ;
        fo_C[i] = uint32_t((u_on[i] ? n : 0) * p.C_dstate_stride) * SZ;
    }
    const int u_lds = 8 * u_q * BCS + u_n;
    const bool padded = N < NP;            // uniform

    // Loads at or past the end of a row are redirected into the row's last elements (always in
    // bounds: L is a multiple of 8, or element by element); the steps they feed are padding with
    // dt' = 0 (and, where a lane's steps may be part padding, u = 0).
    // PEEL: without VEC the partial tile comes after the loop, in code of its own, where a lane holds four
    // states and stages B and C alone: with it in the loop the rank-2 instance spilled 69 registers in fp32 and 20
    // at 16 bits (18 and none so; rank 8, fp16: 108 and 80), 64 x 4,096 channels, L 21, rank 8, dstate 16, fp16: 338 ->
    // 196 us; 24 x 4,096, L 255, rank 8, fp32: 631 -> 580. The other layouts have the registers, and the partial
    // tile's inputs in flight a tile ahead are worth more (2 x 1,536, L 777, dstate 64, fp32: 81 against 87 us).
    constexpr bool PEEL = !VEC && S == 4 && W == 1;
    const int64_t lastE = L - E;
    const char *const ub = reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.u) + b * p.u_batch_stride + dw * p.u_d_stride);
    const char *const db = reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.delta) + b * p.delta_batch_stride + dw * p.delta_d_stride);
    const char *const zb = reinterpret_cast<const char *>(reinterpret_cast<const T *>(p.z) + (p.z ? b * p.z_batch_stride + dw * p.z_d_stride : 0));
    const char *const Bb = reinterpret_cast<const char *>(Bg), *const Cb = reinterpret_cast<const char *>(Cg);
    char *const ob = reinterpret_cast<char *>(reinterpret_cast<T *>(p.out) + (p.out ? b * p.out_batch_stride + dw * p.out_d_stride : 0));
    char *const ozb = reinterpret_cast<char *>(reinterpret_cast<T *>(p.out_z) + (p.out_z ? b * p.out_z_batch_stride + dw * p.out_z_d_stride : 0));
    // Loads run D tiles ahead: rings of D entries (elements, B/C) whose registers stay fixed (the
    // tile loop is unrolled by D below; copying an entry whose loads are in flight would wait for
    // them). D = 2 where the second entry fits in registers (S <= 2); at S = 4 it would spill.
    constexpr int D = S <= 2 ? 2 : 1;
    struct Elems {
        RawVec<T, E> u, d, z;
    };
    auto load_part = [&](int64_t t, Elems &e) {   // of a partial tile, element by element
        e = {};
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t eo = uint32_t(t + es + i < L ? t + es + i : L - 1) * SZ;
            set_raw<T, E>(e.u, i, load_elem<T>(ub, fo_u + eo));
            set_raw<T, E>(e.d, i, load_elem<T>(db, fo_d + eo));
            if (zp) set_raw<T, E>(e.z, i, load_elem<T>(zb, fo_z + eo));
        }
    };
    auto load_elems = [&](int64_t t, Elems &e) {
        if constexpr (!VEC) {
            if (t + kT <= L) {             // uniform: a whole tile
                const int64_t so = t * SZ;
                const uint32_t eo = uint32_t(es) * SZ;
                e.u = load_any<T, E>(ub + so, fo_u + eo);
                e.d = load_any<T, E>(db + so, fo_d + eo);
                if (zp) e.z = load_any<T, E>(zb + so, fo_z + eo);
                else e.z = {};
            } else if (!PEEL && t < L) {
                load_part(t, e);
            }
            return;
        }
        uint32_t eo, so;
        if (t + kT <= L) {                 // uniform: a whole tile
            eo = uint32_t(es) * SZ;
            so = uint32_t(t) * SZ;
        } else {
            eo = uint32_t(t + es < lastE ? t + es : lastE) * SZ;
            so = 0;
        }
        e.u = buffer_load_rawn<T, E>(rs_u, fo_u + eo, so);
        e.d = buffer_load_rawn<T, E>(rs_d, fo_d + eo, so);
        if (zp) e.z = buffer_load_rawn<T, E>(rs_z, fo_z + eo, so);
        else e.z = {};
    };
    struct BCs {
        RawVec<T, 8> b[NU], c[NU];
    };
    auto load_bc = [&](int64_t t0, BCs &r) {
        if (t0 + kT <= L) {                // uniform: a whole tile
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                if constexpr (VEC) {
                    const uint32_t so = uint32_t(t0) * SZ;
                    r.b[i] = buffer_load_rawn<T, 8>(rs_B, fo_B[i] + uint32_t(8 * u_q) * SZ, so);
                    r.c[i] = buffer_load_rawn<T, 8>(rs_C, fo_C[i] + uint32_t(8 * u_q) * SZ, so);
                } else {
                    const int64_t so = t0 * SZ;
                    r.b[i] = load_any<T, 8>(Bb + so, fo_B[i] + uint32_t(8 * u_q) * SZ);
                    r.c[i] = load_any<T, 8>(Cb + so, fo_C[i] + uint32_t(8 * u_q) * SZ);
                }
            }
        } else if constexpr (VEC) {        // the last, partial tile
            const int64_t st = t0 + 8 * u_q;
            const uint32_t o = uint32_t(st < L ? st : L - 8) * SZ;
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                r.b[i] = buffer_load_rawn<T, 8>(rs_B, fo_B[i] + o, 0);
                r.c[i] = buffer_load_rawn<T, 8>(rs_C, fo_C[i] + o, 0);
                if (st >= L) r.b[i] = r.c[i] = {};
            }
        }                                  // without VEC stage_part loads that tile
        if (padded) {
#pragma unroll
            for (int i = 0; i < NU; ++i)
                if (!u_on[i]) r.b[i] = r.c[i] = {};
        }
    };
    // Tile rows [step][B states | C states] as float32 (zeros for padded states and past L).
    auto stage_part = [&](int64_t t0) {    // the partial tile, element by element
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            uint32_t vb[8], vc[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t st = t0 + 8 * u_q + e;
                const uint32_t o = uint32_t(st < L ? st : L - 1) * SZ;
                vb[e] = load_elem<T>(Bb, fo_B[i] + o);
                vc[e] = load_elem<T>(Cb, fo_C[i] + o);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool on = u_on[i] && t0 + 8 * u_q + e < L;
                sBC[u_lds + 16 * W * i + e * BCS] = on ? elem_f32<T>(vb[e]) : 0.f;
                sBC[u_lds + 16 * W * i + e * BCS + NP] = on ? elem_f32<T>(vc[e]) : 0.f;
            }
        }
    };
    auto stage_bc = [&](const BCs &r, int64_t t0) {
        if constexpr (!VEC && !PEEL) {
            if (t0 + kT > L) {             // uniform
                stage_part(t0);
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            float vb[8], vc[8];
            unpack_raw<T, 8>(r.b[i], vb);
            unpack_raw<T, 8>(r.c[i], vc);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sBC[u_lds + 16 * W * i + e * BCS] = vb[e];
                sBC[u_lds + 16 * W * i + e * BCS + NP] = vc[e];
            }
        }
    };
    auto pin = [&](Elems &e, BCs &r) __attribute__((always_inline)) {
        pin_raw(e.u);
        pin_raw(e.d);
        pin_raw(e.z);
        if constexpr (!VEC) {
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                pin_raw(r.b[i]);
                pin_raw(r.c[i]);
            }
        }
    };
    Elems e0, e1;
    BCs b0, b1;
    const int64_t Lt = PEEL ? L - L % kT : L;   // end of the loop's tiles
    if (!PEEL || Lt > 0) {
        load_elems(0, e0);
        if (D == 2) load_elems(kT, e1);
        load_bc(0, b0);
        stage_bc(b0, 0);
        pin(e0, b0);
        if (D == 2) load_bc(kT, b1);
    }

    // Tile t0: its elements in ec, its B/C (already staged) in bc, the next tile's B/C in bn (the
    // same entry as bc when D = 1: loaded at the top of the tile, staged at its end). TAIL: PEEL's partial
    // tile, which nothing follows.
    auto tile = [&](auto tail_c, const int64_t t0, Elems &ec, BCs &bc, Elems &en, BCs &bn) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail_c)::value, WHOLE = PEEL && !TAIL;
        const int64_t t1 = t0 + kT;
        // This lane's elements exist: all or none of them where L is a multiple of E.
        auto ev = [&](int i) { return VEC ? t0 + es < L : WHOLE || t0 + es + i < L; };
        float uu[E], dd[E], zz[E];
        unpack_raw<T, E>(ec.u, uu);
        unpack_raw<T, E>(ec.d, dd);
        unpack_raw<T, E>(ec.z, zz);
        // Prefetch D tiles ahead into the entries just consumed (clamped addresses: in bounds).
        if constexpr (!TAIL) {
            load_elems(t0 + D * kT, ec);
            load_bc(t0 + D * kT, bc);
        }

        // Prologue: dt' and dt' u of (channel, steps es .. es + E - 1).
        float dtp[E], dup[E];
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const float x = dd[i] + bias;
            dtp[i] = softplus ? softplus_fast(x) : x;
            if (!ev(i)) {                  // padded steps of a last, partial tile
                dtp[i] = 0.f;
                if constexpr (!VEC) uu[i] = 0.f;
            }
            dup[i] = dtp[i] * uu[i];
        }
#pragma unroll
        for (int i = 0; i < E; i += 2) {
            *reinterpret_cast<float2 *>(&sDt[cw * kPad + es + i]) = make_float2(dtp[i], dtp[i + 1]);
            *reinterpret_cast<float2 *>(&sDu[cw * kPad + es + i]) = make_float2(dup[i], dup[i + 1]);
        }
        __syncthreads();
        if (ckp) put_ck(t0 / 16);

        // Scan: 32 steps in groups of 4. The decay factors and the input terms of a group do not
        // depend on the state and are formed first; then the coupled updates run in order.
        float yp[kT];
        static_for<0, kT / 4>([&](auto G4) {
            constexpr int s4 = decltype(G4)::value;
            if constexpr (s4 == 4) {
                if (ckp && t0 + 16 < L) put_ck(t0 / 16 + 1);
            }
            const float4 dt4 = *reinterpret_cast<const float4 *>(&sDt[cw * kPad + 4 * s4]);
            const float4 du4 = *reinterpret_cast<const float4 *>(&sDu[cw * kPad + 4 * s4]);
            const float dts[4] = {dt4.x, dt4.y, dt4.z, dt4.w};
            const float dus[4] = {du4.x, du4.y, du4.z, du4.w};
            float av[4][S], bu[4][S], cv[4][S];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = 4 * s4 + j;
                float bv[S];
                lds_read_vec<S>(&sBC[t * BCS + k * S], bv);
                lds_read_vec<S>(&sBC[t * BCS + NP + k * S], cv[j]);
                if constexpr (DX) cum_dt += dts[j];   // steps past L have dt' = 0
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    av[j][s] = decay_exp2(dts[j], A2[s]);
                    bu[j][s] = dus[j] * bv[s];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float q[RR], y = 0.f;
                if constexpr (XK) {
                    // h_t = hb + P q with hb = a h_{t-1} + dt' u B and q = dt' gq; the next step's
                    // lane partial of Q h_t as X + K q, where X = Q hb needs only h_{t-1} (off the
                    // serial chain) and K = Q P over the lane's states.
                    float hb[S], X[R];
#pragma unroll
                    for (int s = 0; s < S; ++s) hb[s] = __builtin_fmaf(av[j][s], h[s], bu[j][s]);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        X[r] = Qr[r][0] * hb[0];
#pragma unroll
                        for (int s = 1; s < S; ++s) X[r] = __builtin_fmaf(Qr[r][s], hb[s], X[r]);
                        q[r] = gq[r] * dts[j];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        float acc = X[r];
#pragma unroll
                        for (int r2 = 0; r2 < R; ++r2) acc = __builtin_fmaf(Kr[r][r2], q[r2], acc);
                        gq[r] = group_sum<LPR>(acc);
                    }
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        float w = hb[s];
#pragma unroll
                        for (int r = 0; r < R; ++r) w = __builtin_fmaf(Pr[s][r], q[r], w);
                        h[s] = w;
                        y = s == 0 ? cv[j][0] * h[0] : __builtin_fmaf(cv[j][s], h[s], y);
                    }
                } else if constexpr (TS) {
#pragma unroll
                    for (int t = 0; t < R; ++t) {
                        q[t] = Qr[t][0] * h[0];
#pragma unroll
                        for (int s = 1; s < S; ++s) q[t] = __builtin_fmaf(Qr[t][s], h[s], q[t]);
                    }
                    lane_sums<LPR, R>(q);
#pragma unroll
                    for (int t = 0; t < R; ++t) q[t] *= dts[j];
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        float w = bu[j][s];
#pragma unroll
                        for (int t = 0; t < R; ++t) w = __builtin_fmaf(Pr[s][t], q[t], w);
                        h[s] = __builtin_fmaf(av[j][s], h[s], w);
                        y = s == 0 ? cv[j][0] * h[0] : __builtin_fmaf(cv[j][s], h[s], y);
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        float acc = Qr[r][0] * h[0];
#pragma unroll
                        for (int s = 1; s < S; ++s) acc = __builtin_fmaf(Qr[r][s], h[s], acc);
                        q[r] = group_sum<LPR>(acc) * dts[j];
                    }
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        float w = bu[j][s];
#pragma unroll
                        for (int r = 0; r < R; ++r) w = __builtin_fmaf(Pr[s][r], q[r], w);
                        h[s] = __builtin_fmaf(av[j][s], h[s], w);
                        y = s == 0 ? cv[j][0] * h[0] : __builtin_fmaf(cv[j][s], h[s], y);
                    }
                }
                yp[4 * s4 + j] = y;
            }
        });
        __syncthreads();                   // sDt / sDu / sBC reads done: sY and sBC are rewritten

#pragma unroll
        for (int t = 0; t < kT; t += 4)
            *reinterpret_cast<float4 *>(&sY[(cw * LPR + k) * kPad + t]) = make_float4(yp[t], yp[t + 1], yp[t + 2], yp[t + 3]);
        if (!TAIL && t1 < Lt) stage_bc(bn, t1);
        // The next tile's inputs are taken as read here, where they have long arrived: at their first use
        // (or, B and C, at the next loads into their registers) the wait for them would be one for the
        // stores below or for the loads just issued as well (2,048 channels, L 30,001, dstate 64, rows of
        // any alignment: 3.7 -> 2.8 ms). Not where a lane's four states spill with rank 8 in fp32: aligned rows,
        // dstate 32, 2 x 4,096 channels, L 2,048: 768 us with it, 756 without (16 x 4,096, L 512: 1,112 and 1,093).
        if constexpr (!TAIL && !(VEC && S == 4 && R == 8 && SZ == 4)) pin(en, bn);
        __syncthreads();

        // Epilogue: y of (channel, steps es .. es + E - 1) = the LPR partials, added in lane order.
        float y[E];
#pragma unroll
        for (int i = 0; i < E; i += 2) {
            float2 acc = *reinterpret_cast<const float2 *>(&sY[(cw * LPR) * kPad + es + i]);
#pragma unroll
            for (int kk = 1; kk < LPR; ++kk) {
                const float2 v = *reinterpret_cast<const float2 *>(&sY[(cw * LPR + kk) * kPad + es + i]);
                acc.x += v.x;
                acc.y += v.y;
            }
            y[i] = acc.x;
            y[i + 1] = acc.y;
        }
        if (active && ev(0)) {
            float o[E];
#pragma unroll
            for (int i = 0; i < E; ++i) o[i] = p.D ? __builtin_fmaf(Dv, uu[i], y[i]) : y[i];
            auto put = [&](auto rs, char *base, uint32_t off) __attribute__((always_inline)) {
                if constexpr (VEC) {
                    buffer_store_vecn<T, E>(rs, off, uint32_t(t0) * SZ, o);
                } else if (WHOLE || (!TAIL && t1 <= L)) {   // uniform
                    store_any<T, E>(base + t0 * SZ, off, o);
                } else {
#pragma unroll
                    for (int i = 0; i < E; ++i)
                        if (ev(i)) store_elem<T>(base + t0 * SZ, off + uint32_t(i) * SZ, o[i]);
                }
            };
            if (p.out) put(rs_o, ob, fo_o);
            if (zp) {
#pragma unroll
                for (int i = 0; i < E; ++i) o[i] *= silu_fast(zz[i]);
                put(rs_oz, ozb, fo_oz);
            }
        }
        if (active && p.chunk_states) {
            const int64_t tend = t1 < L ? t1 : L;
            if (tend % MM_SCAN_CHUNK == 0 || tend == L) {
                const int64_t c = (tend - 1) / MM_SCAN_CHUNK;
                float *cs = p.chunk_states + ((b * p.dim + d) * n_chunks + c) * 2 * N;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const int n = k * S + s;
                    if (n < N) {
                        cs[2 * n] = DX ? __builtin_amdgcn_exp2f(A2[s] * cum_dt) : 1.f;
                        cs[2 * n + 1] = h[s];
                    }
                }
            }
        }
        __syncthreads();                   // sY reads done before the next prologue overwrites sX
    };
    constexpr std::false_type kLoop{};
    if constexpr (D == 2) {
        for (int64_t t0 = 0; t0 < Lt; t0 += 2 * kT) {
            tile(kLoop, t0, e0, b0, e1, b1);
            if (t0 + kT < Lt) tile(kLoop, t0 + kT, e1, b1, e0, b0);
        }
    } else {
        for (int64_t t0 = 0; t0 < Lt; t0 += kT) tile(kLoop, t0, e0, b0, e0, b0);
    }
    if constexpr (PEEL) {
        if (Lt < L) {                      // uniform; the loop's last barrier stands behind its reads of sBC
            load_part(Lt, e0);
            stage_part(Lt);
            tile(std::true_type{}, Lt, e0, b0, e0, b0);
        }
    }
    if (active && p.last_state) {
        float *ls = p.last_state + (b * p.dim + d) * N;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int n = k * S + s;
            if (n < N) ls[n] = h[s];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// scan_fwd_pq_step<T, LPR>: one time step (seqlen 1) with variable B and C, dstate <= 4 LPR: what the
// Motif module's decode step calls. From the zero state Q h is zero, so the coupling's contribution per
// state, P (Q 0), is the same for every batch row: formed once per lane, it keeps the general
// kernels' result for non-finite P, Q and decays. LPR lanes share a (batch, channel) row, four states
// each, and serve U batch rows with one load of A, P and Q, every row's loads issued before the
// first is used. The call moves little more than the final states, which leave as 16-byte stores of
// consecutive lanes (one lane per row wrote each 64-byte state row in 4-byte pieces). No load stands behind
// a branch or a wait for another, addresses are a uniform base and a 32-bit lane offset, and a contiguous
// row of A comes as one vector (of P and Q, too, in the source; the compiler merges their two forms into one
// set of four-byte loads behind the branch). Bound by the state writes beyond some 16 batch rows. 64 x 4,096
// channels, dstate 16, rank 2, fp16 (20 MB): 45.4 us per call with one lane per row, 14.1 us here (15.7
// with a wait per row, per rank and for B and C); 256 rows: 42 us.
// ------------------------------------------------------------------------------------------------
constexpr int kLanesBlock = 256;
constexpr int kStepBC = 1, kStepAPQ = 2;   // four consecutive states per lane: of B and C, of A, P (rank 2) and Q

template <typename T, int LPR, int U>
__global__ void __launch_bounds__(kLanesBlock)
scan_fwd_pq_step(const mm_scan_fwd_params p, const int64_t ratio, const int32_t vec) {
    constexpr int S = 4, CPB = kLanesBlock / LPR;   // channels per block
    constexpr uint32_t SZ = sizeof(T);
    const int k = threadIdx.x % LPR;       // states 4 k .. 4 k + 3
    const int64_t d0 = int64_t(blockIdx.x) * CPB;
    const int64_t left = p.dim - d0;
    const bool active = int(threadIdx.x / LPR) < left;
    const int dl = active ? int(threadIdx.x / LPR) : int(left) - 1;   // clamped for loads; stores are predicated
    const int N = int(p.dstate);
    const int n0 = S * k;
    int nn[S];
    bool on[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        on[s] = n0 + s < N;
        nn[s] = on[s] ? n0 + s : N - 1;
    }

    // Every load is issued before the first is waited for: no branch around one (without z, u is read in its
    // place), and B and C stay raw words until they are used. Addresses are a uniform base (the batch row's
    // or the block's first channel's) and a 32-bit lane offset, which the host has checked to fit.
    auto base = [&](const void *t, int64_t ds) { return reinterpret_cast<const char *>(t) + d0 * ds * int64_t(SZ); };
    const void *const zsrc = p.z ? p.z : p.u;
    const int64_t zb = p.z ? p.z_batch_stride : p.u_batch_stride, zd = p.z ? p.z_d_stride : p.u_d_stride;
    const char *const up = base(p.u, p.u_d_stride), *const dp = base(p.delta, p.delta_d_stride), *const zp = base(zsrc, zd);
    const uint32_t ou = uint32_t(dl) * uint32_t(p.u_d_stride) * SZ, od = uint32_t(dl) * uint32_t(p.delta_d_stride) * SZ;
    const uint32_t oz = uint32_t(dl) * uint32_t(zd) * SZ;
    uint32_t uv[U], dv[U], zv[U];
    RawVec<T, S> bv[U], cv[U];
    const int64_t b0 = int64_t(blockIdx.y) * U;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int64_t b = (b0 + i < p.batch ? b0 + i : p.batch - 1) * int64_t(SZ);
        uv[i] = load_elem<T>(up + b * p.u_batch_stride, ou);
        dv[i] = load_elem<T>(dp + b * p.delta_batch_stride, od);
        zv[i] = load_elem<T>(zp + b * zb, oz);
    }
    // The channel's group: one for the whole block unless its channels straddle groups.
    const int64_t g0 = p.n_groups == 1 ? 0 : d0 / ratio;
    const uint32_t gl = p.n_groups == 1 ? 0u : uint32_t(d0 - g0 * ratio + dl) / uint32_t(ratio);
    const char *const Bp = reinterpret_cast<const char *>(p.B) + g0 * p.B_group_stride * int64_t(SZ);
    const char *const Cp = reinterpret_cast<const char *>(p.C) + g0 * p.C_group_stride * int64_t(SZ);
    const uint32_t oB = gl * uint32_t(p.B_group_stride) * SZ, oC = gl * uint32_t(p.C_group_stride) * SZ;
    if (vec & kStepBC) {                   // consecutive states (uniform); no padded state in a lane
        const uint32_t n = uint32_t(n0 < N ? n0 : 0) * SZ;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int64_t b = (b0 + i < p.batch ? b0 + i : p.batch - 1) * int64_t(SZ);
            bv[i] = load_any<T, S>(Bp + b * p.B_batch_stride, oB + n);
            cv[i] = load_any<T, S>(Cp + b * p.C_batch_stride, oC + n);
        }
    } else {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int64_t b = (b0 + i < p.batch ? b0 + i : p.batch - 1) * int64_t(SZ);
            bv[i] = cv[i] = {};
#pragma unroll
            for (int s = 0; s < S; ++s) {
                set_raw<T, S>(bv[i], s, load_elem<T>(Bp + b * p.B_batch_stride, oB + uint32_t(nn[s]) * uint32_t(p.B_dstate_stride) * SZ));
                set_raw<T, S>(cv[i], s, load_elem<T>(Cp + b * p.C_batch_stride, oC + uint32_t(nn[s]) * uint32_t(p.C_dstate_stride) * SZ));
            }
        }
    }
    // Then A, D, the bias and two ranks of Q and P at a time (clamped states: in bounds).
    auto f32 = [&](const float *t, uint32_t off) { return __uint_as_float(load_elem<float>(reinterpret_cast<const char *>(t), off)); };
    const float *const Ap = p.A + d0 * p.A_d_stride, *const Qp = p.Q + d0 * p.Q_d_stride, *const Pp = p.P + d0 * p.P_d_stride;
    const uint32_t oA = 4 * uint32_t(dl) * uint32_t(p.A_d_stride), oQ = 4 * uint32_t(dl) * uint32_t(p.Q_d_stride);
    const uint32_t oP = 4 * uint32_t(dl) * uint32_t(p.P_d_stride);
    float A2[S], coup[S] = {0.f, 0.f, 0.f, 0.f};
    uint32_t onQ[S], onP[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        onQ[s] = oQ + 4 * uint32_t(nn[s]) * uint32_t(p.Q_dstate_stride);
        onP[s] = oP + 4 * uint32_t(nn[s]) * uint32_t(p.P_dstate_stride);
    }
    const float Dv = p.D ? f32(p.D + d0, 4 * uint32_t(dl)) : 0.f;
    const float bias = p.delta_bias ? f32(p.delta_bias + d0, 4 * uint32_t(dl)) : 0.f;
    const int rank = int(p.pq_rank);
    float Qv[2][S], Pv[2][S];
    auto load_pq = [&](int r0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = r0 + j < rank ? r0 + j : r0;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                Qv[j][s] = f32(Qp + r * p.Q_r_stride, onQ[s]);
                Pv[j][s] = f32(Pp + r * p.P_r_stride, onP[s]);
            }
        }
    };
    // One vector per lane and row (A) instead of four loads that each touch every line of the rows.
    if (vec & kStepAPQ) {
        const uint32_t n = 4 * uint32_t(n0 < N ? n0 : 0);
        auto four = [&](const float *t, uint32_t off, float *o) {
            const RawVec<float, S> v = load_any<float, S>(reinterpret_cast<const char *>(t), off);
#pragma unroll
            for (int s = 0; s < S; ++s) o[s] = __uint_as_float(v.w[s]);
        };
        four(Ap, oA + n, A2);
        four(Qp, oQ + n, Qv[0]);
        four(Qp + p.Q_r_stride, oQ + n, Qv[1]);
        float p8[2 * S];
        four(Pp, oP + 2 * n, p8);
        four(Pp + S, oP + 2 * n, p8 + S);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            Pv[0][s] = p8[2 * s];
            Pv[1][s] = p8[2 * s + 1];
        }
    } else {
#pragma unroll
        for (int s = 0; s < S; ++s) A2[s] = f32(Ap, oA + 4 * uint32_t(nn[s]) * uint32_t(p.A_dstate_stride));
        load_pq(0);
    }
    for (int r0 = 0; r0 < rank; r0 += 2) {
        if (r0 > 0) load_pq(r0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool has = r0 + j < rank;   // else zeros (a branch would take the loads behind it)
            float q = 0.f;
#pragma unroll
            for (int s = 0; s < S; ++s) q = __builtin_fmaf(has && on[s] ? Qv[j][s] : 0.f, 0.f, q);
            q = group_sum<LPR>(q);
#pragma unroll
            for (int s = 0; s < S; ++s) coup[s] = __builtin_fmaf(has && on[s] ? Pv[j][s] : 0.f, q, coup[s]);
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) A2[s] = on[s] ? A2[s] * kLog2e : 0.f;
    const bool ls_vec = N % S == 0 && reinterpret_cast<uintptr_t>(p.last_state) % 16 == 0;
    const bool write_y = active && k == 0;
    const uint32_t oo = uint32_t(dl) * uint32_t(p.out_d_stride) * SZ, ooz = uint32_t(dl) * uint32_t(p.out_z_d_stride) * SZ;

#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int64_t b = b0 + i;
        if (b >= p.batch) break;           // uniform
        float dt = elem_f32<T>(dv[i]) + bias;
        if (p.delta_softplus) dt = softplus_fast(dt);
        const float uu = elem_f32<T>(uv[i]);
        const float du = dt * uu;
        float h[S], y = 0.f, Bv[S], Cv[S];
        unpack_raw<T, S>(bv[i], Bv);
        unpack_raw<T, S>(cv[i], Cv);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const float w = __builtin_fmaf(dt, coup[s], du * (on[s] ? Bv[s] : 0.f));
            h[s] = __builtin_fmaf(decay_exp2(dt, A2[s]), 0.f, w);
            y = __builtin_fmaf(h[s], on[s] ? Cv[s] : 0.f, y);
        }
        y = group_sum<LPR>(y);
        const float o = p.D ? __builtin_fmaf(Dv, uu, y) : y;
        if (write_y) {
            const int64_t bz = b * int64_t(SZ);
            if (p.out)
                store_elem<T>(reinterpret_cast<char *>(p.out) + d0 * p.out_d_stride * int64_t(SZ) + bz * p.out_batch_stride, oo, o);
            if (p.out_z)
                store_elem<T>(reinterpret_cast<char *>(p.out_z) + d0 * p.out_z_d_stride * int64_t(SZ) + bz * p.out_z_batch_stride, ooz,
                              o * silu_fast(elem_f32<T>(zv[i])));
        }
        if (active && p.last_state) {
            float *ls = p.last_state + (b * p.dim + d0) * N + (dl * N + n0);
            if (ls_vec) {
                if (n0 < N) *reinterpret_cast<float4 *>(ls) = make_float4(h[0], h[1], h[2], h[3]);
            } else {
#pragma unroll
                for (int s = 0; s < S; ++s)
                    if (on[s]) ls[s] = h[s];
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// scan_fwd_pq_lanes<T, LPR, R>: any request with dstate <= 4 LPR -- constant B/C, any strides,
// alignment and length, every output: what neither the tiled nor the one-step kernel takes. LPR lanes
// share a (batch, channel) row, four states each in registers with their A, P and Q, the coupling's R
// sums as DPP butterflies, the next step's inputs in flight during a step.
// ------------------------------------------------------------------------------------------------
template <typename T, int LPR, int R>
__global__ void __launch_bounds__(kLanesBlock)
scan_fwd_pq_lanes(const mm_scan_fwd_params p, const int64_t ratio) {
    constexpr int S = 4;
    const int k = threadIdx.x % LPR;       // states 4 k .. 4 k + 3
    const int64_t d_raw = int64_t(blockIdx.x) * (kLanesBlock / LPR) + threadIdx.x / LPR;
    const int64_t b = blockIdx.y;
    const bool active = d_raw < p.dim;
    const int64_t d = active ? d_raw : p.dim - 1;  // clamped for loads; stores are predicated
    const int64_t g = d / ratio;
    const int64_t L = p.seqlen;
    const int N = int(p.dstate);
    const int rank = int(p.pq_rank);
    const int n0 = S * k;

    float A2[S], Pr[S][R], Qr[R][S], Bc[S], Cc[S];
    const T *Bv[S], *Cv[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int n = n0 + s;
        const bool on = n < N;
        const int nn = on ? n : N - 1;
        A2[s] = on ? p.A[d * p.A_d_stride + n * p.A_dstate_stride] * kLog2e : 0.f;
        Bc[s] = on && !p.is_variable_B ? reinterpret_cast<const float *>(p.B)[d * p.B_d_stride + n * p.B_dstate_stride] : 0.f;
        Cc[s] = on && !p.is_variable_C ? reinterpret_cast<const float *>(p.C)[d * p.C_d_stride + n * p.C_dstate_stride] : 0.f;
        Bv[s] = reinterpret_cast<const T *>(p.B) + b * p.B_batch_stride + g * p.B_group_stride + nn * p.B_dstate_stride;
        Cv[s] = reinterpret_cast<const T *>(p.C) + b * p.C_batch_stride + g * p.C_group_stride + nn * p.C_dstate_stride;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool use = on && r < rank;
            Pr[s][r] = use ? p.P[d * p.P_d_stride + n * p.P_dstate_stride + r * p.P_r_stride] : 0.f;
            Qr[r][s] = use ? p.Q[d * p.Q_d_stride + r * p.Q_r_stride + n * p.Q_dstate_stride] : 0.f;
        }
    }
    const float Dv = p.D ? p.D[d] : 0.f;
    const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
    const int64_t n_chunks = (L + MM_SCAN_CHUNK - 1) / MM_SCAN_CHUNK;
    const T *up = reinterpret_cast<const T *>(p.u) + b * p.u_batch_stride + d * p.u_d_stride;
    const T *dp = reinterpret_cast<const T *>(p.delta) + b * p.delta_batch_stride + d * p.delta_d_stride;
    const T *zp = p.z ? reinterpret_cast<const T *>(p.z) + b * p.z_batch_stride + d * p.z_d_stride : nullptr;
    T *op = p.out ? reinterpret_cast<T *>(p.out) + b * p.out_batch_stride + d * p.out_d_stride : nullptr;
    T *ozp = p.out_z ? reinterpret_cast<T *>(p.out_z) + b * p.out_z_batch_stride + d * p.out_z_d_stride : nullptr;
    struct Step {
        T u, d, z, b[S], c[S];
    };
    auto load = [&](int64_t t) {
        Step x;
        x.u = up[t];
        x.d = dp[t];
        if (zp) x.z = zp[t];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (p.is_variable_B) x.b[s] = Bv[s][t];
            if (p.is_variable_C) x.c[s] = Cv[s][t];
        }
        return x;
    };
    float h[S] = {0.f, 0.f, 0.f, 0.f};
    Step nxt = load(0);
    for (int64_t t = 0; t < L; ++t) {
        const Step x = nxt;
        nxt = load(t + 1 < L ? t + 1 : t);     // in flight during this step
        if (p.tile_states && active && t % 16 == 0) {
            // The state before this 16-step tile, for the backward (states past dstate are 0).
            float *ck = p.tile_states + ((t / 16) * p.batch * p.dim + b * p.dim + d) * 16 + n0;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (n0 + s < 16) ck[s] = h[s];
        }
        float dt = to_f32(x.d) + bias;
        if (p.delta_softplus) dt = softplus_fast(dt);
        const float uu = to_f32(x.u);
        const float du = dt * uu;
        float q[R];                            // dt' (Q h_{t-1})
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float acc = Qr[r][0] * h[0];
#pragma unroll
            for (int s = 1; s < S; ++s) acc = __builtin_fmaf(Qr[r][s], h[s], acc);
            q[r] = group_sum<LPR>(acc) * dt;
        }
        float y = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool on = n0 + s < N;
            float w = du * (p.is_variable_B ? (on ? to_f32(x.b[s]) : 0.f) : Bc[s]);
#pragma unroll
            for (int r = 0; r < R; ++r) w = __builtin_fmaf(Pr[s][r], q[r], w);
            h[s] = __builtin_fmaf(decay_exp2(dt, A2[s]), h[s], w);
            y = __builtin_fmaf(h[s], p.is_variable_C ? (on ? to_f32(x.c[s]) : 0.f) : Cc[s], y);
        }
        y = group_sum<LPR>(y);
        if (active && k == 0) {
            const float o = p.D ? __builtin_fmaf(Dv, uu, y) : y;
            if (op) op[t] = from_f32<T>(o);
            if (ozp) ozp[t] = from_f32<T>(o * silu_fast(to_f32(x.z)));
        }
        if (active && p.chunk_states && ((t + 1) % MM_SCAN_CHUNK == 0 || t == L - 1)) {
            float *cs = p.chunk_states + ((b * p.dim + d) * n_chunks + t / MM_SCAN_CHUNK) * 2 * N;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if (n0 + s < N) {
                    cs[2 * (n0 + s)] = 1.f;
                    cs[2 * (n0 + s) + 1] = h[s];
                }
            }
        }
    }
    if (active && p.last_state) {
        float *ls = p.last_state + (b * p.dim + d) * N + n0;
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (n0 + s < N) ls[s] = h[s];
    }
}

// ------------------------------------------------------------------------------------------------
// dstate past 64 (where no request has tile states) and rows of no step: one lane per (batch, channel)
// row; the row's states in LDS (dstate x 64 floats per
// block, lane-minor so every access is conflict-free), P and Q read through the cache.
// ------------------------------------------------------------------------------------------------
constexpr int kRowBlock = 64;

template <typename T>
__global__ void __launch_bounds__(kRowBlock)
scan_fwd_pq_rowlane(const mm_scan_fwd_params p, const int64_t ratio) {
    extern __shared__ float sH[];          // [dstate][64]
    const int lane = threadIdx.x;
    const int64_t d_raw = int64_t(blockIdx.x) * blockDim.x + lane;
    const int64_t b = blockIdx.y;
    const bool active = d_raw < p.dim;
    const int64_t d = active ? d_raw : p.dim - 1;  // clamped for loads; stores are predicated
    const int64_t g = d / ratio;
    const int64_t L = p.seqlen;
    const int N = int(p.dstate);
    const int rank = int(p.pq_rank);

    const T *up = reinterpret_cast<const T *>(p.u) + b * p.u_batch_stride + d * p.u_d_stride;
    const T *dp = reinterpret_cast<const T *>(p.delta) + b * p.delta_batch_stride + d * p.delta_d_stride;
    const T *zp = p.z ? reinterpret_cast<const T *>(p.z) + b * p.z_batch_stride + d * p.z_d_stride : nullptr;
    T *op = p.out ? reinterpret_cast<T *>(p.out) + b * p.out_batch_stride + d * p.out_d_stride : nullptr;
    T *ozp = p.out_z ? reinterpret_cast<T *>(p.out_z) + b * p.out_z_batch_stride + d * p.out_z_d_stride : nullptr;
    const T *Bv = p.is_variable_B ? reinterpret_cast<const T *>(p.B) + b * p.B_batch_stride + g * p.B_group_stride : nullptr;
    const T *Cv = p.is_variable_C ? reinterpret_cast<const T *>(p.C) + b * p.C_batch_stride + g * p.C_group_stride : nullptr;
    const float *Bc = reinterpret_cast<const float *>(p.B) + d * p.B_d_stride;
    const float *Cc = reinterpret_cast<const float *>(p.C) + d * p.C_d_stride;
    const float *Ad = p.A + d * p.A_d_stride;
    const float *Pd = p.P + d * p.P_d_stride;
    const float *Qd = p.Q + d * p.Q_d_stride;

    for (int n = 0; n < N; ++n) sH[n * kRowBlock + lane] = 0.f;
    const float Dv = p.D ? p.D[d] : 0.f;
    const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
    const int64_t n_chunks = (L + MM_SCAN_CHUNK - 1) / MM_SCAN_CHUNK;

    for (int64_t t = 0; t < L; ++t) {
        float dt = to_f32(dp[t]) + bias;
        if (p.delta_softplus) dt = softplus_fast(dt);
        const float uu = to_f32(up[t]);
        const float du = dt * uu;
        // q = dt' (Q h_{t-1}), from the state before this step.
        float q[kMaxRank];
#pragma unroll
        for (int j = 0; j < kMaxRank; ++j) q[j] = 0.f;
        for (int n = 0; n < N; ++n) {
            const float hn = sH[n * kRowBlock + lane];
#pragma unroll
            for (int j = 0; j < kMaxRank; ++j)
                if (j < rank) q[j] = __builtin_fmaf(Qd[j * p.Q_r_stride + n * p.Q_dstate_stride], hn, q[j]);
        }
#pragma unroll
        for (int j = 0; j < kMaxRank; ++j) q[j] *= dt;
        float y = 0.f;
        for (int n = 0; n < N; ++n) {
            const float bn = Bv ? to_f32(Bv[n * p.B_dstate_stride + t]) : Bc[n * p.B_dstate_stride];
            const float cn = Cv ? to_f32(Cv[n * p.C_dstate_stride + t]) : Cc[n * p.C_dstate_stride];
            float w = du * bn;
#pragma unroll
            for (int j = 0; j < kMaxRank; ++j)
                if (j < rank) w = __builtin_fmaf(Pd[n * p.P_dstate_stride + j * p.P_r_stride], q[j], w);
            const float a = decay_exp2(dt, Ad[n * p.A_dstate_stride] * kLog2e);
            const float hn = __builtin_fmaf(a, sH[n * kRowBlock + lane], w);
            sH[n * kRowBlock + lane] = hn;
            y = __builtin_fmaf(hn, cn, y);
        }
        if (active) {
            const float o = p.D ? __builtin_fmaf(Dv, uu, y) : y;
            if (op) op[t] = from_f32<T>(o);
            if (ozp) ozp[t] = from_f32<T>(o * silu_fast(to_f32(zp[t])));
            if (p.chunk_states && ((t + 1) % MM_SCAN_CHUNK == 0 || t == L - 1)) {
                float *cs = p.chunk_states + ((b * p.dim + d) * n_chunks + t / MM_SCAN_CHUNK) * 2 * N;
                for (int n = 0; n < N; ++n) {
                    cs[2 * n] = 1.f;
                    cs[2 * n + 1] = sH[n * kRowBlock + lane];
                }
            }
        }
    }
    if (active && p.last_state) {
        float *ls = p.last_state + (b * p.dim + d) * N;
        for (int n = 0; n < N; ++n) ls[n] = sH[n * kRowBlock + lane];
    }
}

// ------------------------------------------------------------------------------------------------
// Host side.
// ------------------------------------------------------------------------------------------------
struct TiledShape { int S, LPR; };

// The tiled kernel addresses u, delta, z, out and out_z with 32-bit byte offsets from the first of a
// wave's channel rows (up to 16), and B / C from the (batch, group) base: every offset must fit.
static bool offsets_ok(const mm_scan_fwd_params &p) {
    const int64_t eb = p.itype == MM_FLOAT32 ? 4 : 2;
    const int64_t ch = 15 * std::max({p.u_d_stride, p.delta_d_stride, p.z ? p.z_d_stride : int64_t(0),
                                      p.out ? p.out_d_stride : int64_t(0), p.out_z ? p.out_z_d_stride : int64_t(0)});
    const int64_t bc = (p.dstate - 1) * std::max(p.B_dstate_stride, p.C_dstate_stride);
    return (std::max(ch, bc) + p.seqlen) * eb < (int64_t(1) << 32);
}

// The (S, LPR) of the tiled kernel for this request, or {0, 0} when the request needs the general
// kernel: variable B and C, dstate <= 64, seqlen >= 8, offsets that fit in 32 bits.
static TiledShape tiled_shape(const mm_scan_fwd_params &p) {
    if (!p.is_variable_B || !p.is_variable_C || p.dstate > 64 || p.seqlen < 8 || !offsets_ok(p)) return {0, 0};
    const int64_t ratio = p.dim / p.n_groups;
    auto waves = [&](int lpr) { return p.batch * p.n_groups * ((ratio + 64 / lpr - 1) / (64 / lpr)); };
    const char *forced = getenv("MM_PQ_LPR");
    const int want = forced ? atoi(forced) : 0;
    TiledShape cands[3];
    int nc = 0;
    if (p.dstate <= 16) { cands[nc++] = {4, 4}; cands[nc++] = {2, 8}; cands[nc++] = {1, 16}; }
    else if (p.dstate <= 32) { cands[nc++] = {4, 8}; cands[nc++] = {2, 16}; }
    else { cands[nc++] = {4, 16}; }
    for (int i = 0; i < nc; ++i)
        if (cands[i].LPR == want) return cands[i];
    // Measured (fp16, rank 2, L 2048, 2,048-5,120 channels, batch 1-8, on 1,024 SIMDs). 16 lanes per
    // channel add a butterfly stage to every reduction: they win only while their waves fit one per
    // SIMD (dstate 16: 0.191 against 0.214 ms with 8 lanes; dstate 32: 0.244 against 0.31 ms with
    // 8 lanes of 4 states), and lose beyond (dstate 16: 0.58 against 0.30 ms at two waves of 8 lanes
    // per SIMD; dstate 32: 0.60 against 0.47 ms at 1.5). At dstate 16, 8 lanes of 2 states stay the
    // fastest up to 2.5 of their waves per SIMD (0.30 ms at two, 0.40 ms at 2.5 against 0.45 ms with
    // 4 lanes); past that the 4-lane layout's half as many waves win (0.45 against 0.55 ms at 3).
    // Without a coupling the lanes of a channel only meet in y: bf16, L 2048, 2,048 channels x batch 4
    // (1,024 waves of 8 lanes): 0.183 against 0.199 ms at dstate 32, equal at dstate 8; with 1,536 such
    // waves 0.150 against 0.138 and 0.134 against 0.094 ms. 4 lanes stay behind 8 up to 2.5 waves of 8 per
    // SIMD (dstate 8, L 2048: 0.296 against 0.244 ms) and win past that on aligned rows (4 against 8 lanes,
    // dstate 4 and 12 alike, us: 3 per SIMD, L 512, fp16 77 90, fp32 77 84; 4: 80 106, 82 100; 5: 119 118,
    // 129 142; 16: 303 339, 313 406; 32, L 8: 44 53, 44 66). Unaligned rows keep 8: there the partial tile costs a
    // lane of four states more (32 per SIMD, L 63, fp32: 134 against 126).
    const int64_t simds = device_simds();
    if (nc == 1) return cands[0];
    if (waves(16) <= (p.P ? 1 : 2) * simds) return cands[nc - 1];
    if (nc == 2) return cands[0];
    if (!p.P && !fwd_vector_ok(&p)) return cands[1];
    return 2 * waves(8) <= 5 * simds ? cands[1] : cands[0];
}

template <typename T, int S, int LPR, int R, bool VEC>
int launch_tiled_sr(const mm_scan_fwd_params &p, hipStream_t s) {
    constexpr int CPB = 64 / LPR * waves_sharing(S * LPR);   // channels per workgroup
    const int64_t ratio = p.dim / p.n_groups;
    const int64_t bpg = (ratio + CPB - 1) / CPB;
    dim3 grid(unsigned(bpg * p.n_groups), unsigned(p.batch));
    hipLaunchKernelGGL((scan_fwd_pq_tiled<T, S, LPR, R, VEC>), grid, dim3(64 * waves_sharing(S * LPR)), 0, s, p, ratio, int32_t(bpg));
    return launch_status("scan_fwd_pq_tiled");
}

template <typename T, int S, int LPR, bool VEC>
int launch_tiled_v(const mm_scan_fwd_params &p, hipStream_t s) {
    if (!p.P) return launch_tiled_sr<T, S, LPR, 0, VEC>(p, s);
    if (p.pq_rank <= 2) return launch_tiled_sr<T, S, LPR, 2, VEC>(p, s);
    if (p.pq_rank <= 4) return launch_tiled_sr<T, S, LPR, 4, VEC>(p, s);
    return launch_tiled_sr<T, S, LPR, 8, VEC>(p, s);
}
template <typename T, int S, int LPR>
int launch_tiled_s(const mm_scan_fwd_params &p, hipStream_t s) {
    return fwd_vector_ok(&p) ? launch_tiled_v<T, S, LPR, true>(p, s) : launch_tiled_v<T, S, LPR, false>(p, s);
}

// The step kernel's 32-bit lane offsets from a block's first channel (up to 63 channels behind it, in up
// to as many groups) must fit.
static bool step_offsets_ok(const mm_scan_fwd_params &p) {
    const int64_t eb = p.itype == MM_FLOAT32 ? 4 : 2, n = p.dstate - 1, lim = int64_t(1) << 32;
    auto fits = [&](int64_t ds, int64_t ns, int64_t bytes) { return ds >= 0 && ns >= 0 && (63 * ds + n * ns + 4) * bytes < lim; };
    return p.dim < (int64_t(1) << 31) && fits(p.u_d_stride, 0, eb) && fits(p.delta_d_stride, 0, eb) &&
           fits(p.z ? p.z_d_stride : 0, 0, eb) && fits(p.out ? p.out_d_stride : 0, 0, eb) &&
           fits(p.out_z ? p.out_z_d_stride : 0, 0, eb) && fits(p.B_group_stride, p.B_dstate_stride, eb) &&
           fits(p.C_group_stride, p.C_dstate_stride, eb) && fits(p.A_d_stride, p.A_dstate_stride, 4) &&
           fits(p.P_d_stride, p.P_dstate_stride, 4) && fits(p.Q_d_stride, p.Q_dstate_stride, 4);
}

// One-step requests with variable B and C that write no chunk or tile states take the step kernel:
// four batch rows per workgroup where that leaves at least one workgroup per SIMD, else one. It reads a
// first rank of P and Q before it looks at the rank: at rank 0, where P and Q hold no element,
// scan_fwd_pq_lanes serves the call, whose every access stands behind r < rank.
template <typename T, int LPR>
int launch_lanes(const mm_scan_fwd_params &p, hipStream_t s) {
    const int64_t dblk = (p.dim + kLanesBlock / LPR - 1) / (kLanesBlock / LPR), ratio = p.dim / p.n_groups;
    const dim3 grid(unsigned(dblk), unsigned(p.batch)), block(kLanesBlock);
    if (p.seqlen == 1 && p.pq_rank >= 1 && p.is_variable_B && p.is_variable_C && !p.chunk_states && !p.tile_states && step_offsets_ok(p)) {
        int32_t vec = 0;
        if (p.dstate % 4 == 0 && p.B_dstate_stride == 1 && p.C_dstate_stride == 1) vec |= kStepBC;
        if (p.dstate % 4 == 0 && p.A_dstate_stride == 1 && p.Q_dstate_stride == 1 && p.pq_rank == 2 &&
            p.P_r_stride == 1 && p.P_dstate_stride == 2)
            vec |= kStepAPQ;
        if (dblk * ((p.batch + 3) / 4) >= device_simds())
            hipLaunchKernelGGL((scan_fwd_pq_step<T, LPR, 4>), dim3(unsigned(dblk), unsigned((p.batch + 3) / 4)), block,
                               0, s, p, ratio, vec);
        else
            hipLaunchKernelGGL((scan_fwd_pq_step<T, LPR, 1>), grid, block, 0, s, p, ratio, vec);
        return launch_status("scan_fwd_pq_step");
    }
    if (p.pq_rank <= 2) hipLaunchKernelGGL((scan_fwd_pq_lanes<T, LPR, 2>), grid, block, 0, s, p, ratio);
    else hipLaunchKernelGGL((scan_fwd_pq_lanes<T, LPR, 8>), grid, block, 0, s, p, ratio);
    return launch_status("scan_fwd_pq_lanes");
}

template <typename T>
int launch_rowlane(const mm_scan_fwd_params &p, hipStream_t s) {
    if (p.seqlen > 0) {
        if (p.dstate <= 16) return launch_lanes<T, 4>(p, s);
        if (p.dstate <= 32) return launch_lanes<T, 8>(p, s);
        if (p.dstate <= 64) return launch_lanes<T, 16>(p, s);
    }
    dim3 grid(unsigned((p.dim + kRowBlock - 1) / kRowBlock), unsigned(p.batch));
    const size_t lds = size_t(p.dstate) * kRowBlock * sizeof(float);  // <= 64 KB at dstate 256
    hipLaunchKernelGGL((scan_fwd_pq_rowlane<T>), grid, dim3(kRowBlock), lds, s, p, p.dim / p.n_groups);
    return launch_status("scan_fwd_pq_rowlane");
}

}  // namespace pq

template <typename T>
int launch_pq(const mm_scan_fwd_params &p, hipStream_t s) {
    const pq::TiledShape sh = pq::tiled_shape(p);
    if (sh.LPR == 4) return pq::launch_tiled_s<T, 4, 4>(p, s);
    if (sh.LPR == 8) return sh.S == 4 ? pq::launch_tiled_s<T, 4, 8>(p, s) : pq::launch_tiled_s<T, 2, 8>(p, s);
    if (sh.LPR == 16) {
        if (sh.S == 4) return pq::launch_tiled_s<T, 4, 16>(p, s);
        if (sh.S == 2) return pq::launch_tiled_s<T, 2, 16>(p, s);
        return pq::launch_tiled_s<T, 1, 16>(p, s);
    }
    return pq::launch_rowlane<T>(p, s);   // with P and Q (diag_via_pq_fwd requires a tiled shape)
}

template int launch_pq<MM_PQ_TYPE>(const mm_scan_fwd_params &, hipStream_t);

#ifdef MM_PQ_COMMON

// ------------------------------------------------------------------------------------------------
// The diagonal scan on the P/Q kernels without a coupling: requests the dstate-16 kernels do not take
// (forwards with dstate below 16, or 17 to 64; backwards also of odd lengths and unaligned rows), variable
// B and C, run several times faster this way than on the general kernels.
namespace {
// MM_DIAG_VIA_PQ=0 keeps such requests on the general kernels (read per call, for the tests).
bool diag_pq_enabled() {
    const char *e = getenv("MM_DIAG_VIA_PQ");
    return !(e && e[0] == '0');
}

// Inference rows shorter than half a tile, odd or unaligned, of many channels: the tiled kernel stages a tile's
// worth of B and C element by element whatever the length, the row-per-lane kernel's work grows with length
// times dstate (us, row-per-lane against tiled):
//              16 x 4,096 channels                        64 x 4,096 channels
//              L 8          L 9          L 13             L 8          L 9          L 13         L 15
//   fp16  4    14.2 22.2    19.8 22.4    22.6 22.9        28.3 80.1    39.4 81.5    50.7 84.1    56.3 84.1
//         8    19.0 22.2    26.4 22.4                     39.3 80.5    54.2 81.8    68.8 84.4    76.7 84.2
//         12   24.1 22.2    33.5 22.5                     49.0 80.6    67.8 82.1    86.1 84.7    96.2 84.7
//         32                                              116  101
//   fp32  4    11.5 20.4    16.7 20.5    19.8 21.2        23.7 73.5    33.6 74.0    43.0 75.6    48.4 75.8
//         8    13.8 20.5    20.4 20.6    23.8 21.3        30.0 73.7    42.4 74.1    52.3 75.9    59.5 75.8
//         12   16.6 20.6    24.6 20.8    28.8 21.5        34.6 74.3    49.5 74.7    61.1 75.8    68.5 75.9
//         32                                              78.6 102     110  104
// and with fewer rows the tiled kernel wins (8 x 4,096, dstate 8, L 9, fp16: 25.9 against 12.6).
bool short_rows(const mm_scan_fwd_params &p) {
    if (p.seqlen >= 16 || p.chunk_states || p.tile_states || fwd_vector_ok(&p)) return false;
    const int64_t waves = p.batch * p.dim / 8 / device_simds(), work = p.seqlen * p.dstate;   // eight-lane waves per SIMD
    const bool f32 = p.itype == MM_FLOAT32;
    if (waves >= 32) return work <= (!f32 ? 150 : p.seqlen == 8 ? 256 : 200);
    return waves >= 8 && work <= (f32 ? 100 : p.seqlen == 8 ? 64 : 44);
}
}  // namespace

bool diag_via_pq_fwd(const mm_scan_fwd_params &p) {
    // The tiled P/Q kernel then writes the chunk states in the diagonal form (DX), and the tile
    // states below dstate 16 (states past dstate stay 0), which the backward reads.
    if (p.P || p.dstate == 16 || p.dstate > 64 || (p.tile_states && p.dstate > 16) || !diag_pq_enabled())
        return false;
    if (short_rows(p)) return false;
    return pq::tiled_shape(p).LPR != 0;
}

bool diag_lanes_bwd(const mm_scan_bwd_params &p) {
    return !p.P && diag_pq_enabled() && !bwd_tiled_ok(p) && bwd_lanes_ok(p);
}

#endif  // MM_PQ_COMMON

}  // namespace mm
