// mm_internal.h -- declarations shared between the translation units of libmm_scan.so.
#pragma once

#include <hip/hip_runtime.h>

#include "mm_scan.h"

namespace mm {

// Records the launch status of the kernel just enqueued (hipGetLastError) and the error text.
int launch_status(const char *what);
// Records `msg` as the thread's last error and returns `code`.
int set_error(int code, const char *msg);

// True when every activation row start (u, delta, z, out, out_z, variable B/C) is 16-byte aligned
// and seqlen is a multiple of 8, so rows can be moved in 16-byte vectors.
bool fwd_vector_ok(const mm_scan_fwd_params *p);

// Tiled forward kernel (mm_scan_tiled.hip). Returns MM_ERR_UNSUPPORTED, without launching,
// when the request falls outside the shapes that kernel covers; the caller then uses the
// lane-per-row kernel.
template <typename T>
int try_launch_tiled(const mm_scan_fwd_params &p, hipStream_t stream);

// Number of sequence segments the dstate-16 kernels use for `p` (1: a single pass), and the
// workspace bytes that takes (mm_scan_tiled.hip).
int64_t segment_count(const mm_scan_fwd_params &p);
bool tile_states_ok(const mm_scan_fwd_params &p);
// The states before every 16-step tile, alone, into p.tile_states (the backward's checkpoints when
// the forward did not save them); MM_ERR_UNSUPPORTED without launching when tile_states_ok fails.
template <typename T>
int launch_states_only(const mm_scan_fwd_params &p, hipStream_t stream);
int64_t segment_workspace_bytes(const mm_scan_fwd_params &p, int64_t n_seg);

// SIMDs of the current device (4 per CU; cached per device), 1024 when it cannot be queried
// (mm_scan_tiled.hip).
int64_t device_simds();
// Whether a diagonal dstate-16 forward runs on the kernel for any length and row alignment.
bool ragged_route(const mm_scan_fwd_params &p);

// Forward scan with the low-rank P/Q coupling (mm_scan_pq.hip): the tiled kernel when the request
// fits it, else the lane-per-row kernel.
template <typename T>
int launch_pq(const mm_scan_fwd_params &p, hipStream_t stream);

// The diagonal scan on the P/Q kernels without a coupling, for requests the dstate-16 kernels do not
// take: diag_via_pq_fwd tells whether a forward goes that way (dstate != 16 up to 64, launch_pq then
// takes it), diag_lanes_bwd whether a backward does (dstate <= 64, scan_bwd_lanes).
bool diag_via_pq_fwd(const mm_scan_fwd_params &p);
bool diag_lanes_bwd(const mm_scan_bwd_params &p);

// Backward (mm_scan_bwd.hip): clears the accumulated gradients and launches the backward kernels
// on `stream`; bwd_workspace_bytes() is the scratch it uses best, bwd_workspace_min_bytes() the
// least it accepts (with tile states: without the segment carries, every unit then a whole row).
template <typename T>
int launch_bwd(const mm_scan_bwd_params &p, hipStream_t stream);
int64_t bwd_workspace_bytes(const mm_scan_bwd_params &p);
int64_t bwd_workspace_min_bytes(const mm_scan_bwd_params &p);
// Whether the dstate-16 diagonal backward takes the request, whole or split into groups of 16 states.
bool bwd_tiled_ok(const mm_scan_bwd_params &p);

// Backward with the low-rank P/Q coupling, dstate <= 64 (mm_scan_bwd_lanes.hip): bwd_lanes_ok() tells
// whether the request fits the kernel; launch_bwd_lanes() runs it on the batch rows of `p` with the
// checkpoints `ck` ([tile][ck_batch][dim][bwd_lanes_np()]) and the dB / dC partial slabs
// ([dim / 16 / n_groups][batch][group][bwd_lanes_np()][L up to a multiple of 4]); the caller clears
// the accumulated gradients first, launches bwd_lanes_batch() rows at a time and reduces the slabs.
bool bwd_lanes_ok(const mm_scan_bwd_params &p);
int bwd_lanes_np(const mm_scan_bwd_params &p);
int64_t bwd_lanes_batch(const mm_scan_bwd_params &p);
template <typename T>
int launch_bwd_lanes(const mm_scan_bwd_params &p, hipStream_t stream, float *ck, int64_t ck_batch, float *partB,
                     float *partC);
// The P/Q backward for the other shapes (mm_scan_pq_bwd.hip; dstate up to 256, constant B or C, any length and channel
// count): one lane per state, checkpoints `ck` of pq_general_ck_floats() floats, float32 atomics.
template <typename T>
int launch_pq_general(const mm_scan_bwd_params &p, hipStream_t stream, float *ck, float *partB, float *partC);
int64_t pq_general_ck_floats(const mm_scan_bwd_params &p);
int pq_general_rows_per_block(const mm_scan_bwd_params &p);

// The general backward kernels' dB/dC partial slabs (mm_scan_bwd.hip): when the rows a workgroup
// holds (rpb) all belong to one (batch, group) -- channels per group a multiple of rpb -- and the
// slabs stay under 4 GiB, each workgroup stores its sums over its rows into its own slab
// [block][batch][group][dstate][seqlen] and gen_slab_reduce adds the blocks in order (no atomics);
// gen_slab_floats() is 0 otherwise (the kernels then add with float32 atomics).
int64_t gen_slab_floats(const mm_scan_bwd_params &p, int64_t rpb);
int launch_gen_slab_reduce(const mm_scan_bwd_params &p, hipStream_t stream, const float *partB, const float *partC,
                           int64_t rpb);

}  // namespace mm
