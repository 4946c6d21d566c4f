// Kernel argument blocks and launcher declarations (internal to libflexatt).
#pragma once
#include <hip/hip_runtime.h>

#include "flexatt_device.h"

namespace flexatt {

struct FwdArgs {
  View q, k, v;
  MutView o;
  float* lse;
  Shape p;
  int nqt;    // number of query tiles (set by the launcher)
  int gpack;  // query heads per workgroup (set by the launcher)
  int bstride;  // block-sparse maps: bytes per wave's block-map row in dynamic LDS (set by the launcher)
};

struct DeltaArgs {
  View o, dout;
  float* delta;
  int B, H, S, D;
  int* zero;  // when set: 4 queue counters the pass clears for the kernels after it
};

struct BwdArgs {
  View q, k, v, dout;
  const float* lse;
  const float* delta;
  MutView dq, dk, dv;
  Shape p;
  int ntiles;  // number of row tiles of the kernel's grid (set by the launcher)
  // dQ with Delta computed in the kernel (bwd_q only): O, and where Delta is
  // written for the dK/dV kernel; delta_out == nullptr: Delta is read from delta.
  View o;
  float* delta_out;
  // Staged dS (D = 128 fp16/bf16): the workspace the dK/dV kernel writes and
  // the dQ kernel reads, and the units stored per query head (the layout is
  // described with ds_tile_offset); ds == nullptr: not staged.
  char* ds;
  int64_t ds_head;
  // Work queue (staged path): queue == nullptr keeps the static work order;
  // otherwise workgroups from nstatic on take their slot from the counter.
  int* queue;
  int nstatic;
  // Staged dK/dV with each KV block's query tiles shared by nparts workgroups:
  // their fp32 sums [part][dK, dV][B * Hkv * Skv][D] (nparts == 1: none)
  float* part;
  int nparts;
};

// Split-KV forward (fwd_split.hip): partials in the caller's workspace, none
// with one split per row tile.
struct DecodeArgs {
  View q, k, v;
  MutView o;
  float* lse;
  float* part_o;    // [B * Hq * Sq][nsplit][D], O of each partial / its row sums
  float* part_lse;  // [B * Hq * Sq][nsplit], LSE of each partial in log2 units
  Shape p;
  int nsplit;  // workgroups per row tile
  int chunk;   // 32-row KV tiles per workgroup (nsplit > 1)
  int nw;      // waves per workgroup with one split (4 or 8; D = 256: 4)
  int nrt;     // 32-row tiles of packed query rows per (b, hkv) (set by the launcher)
  int plain;   // workgroups in plain order instead of by XCD (set by the launcher)
};

// Backward in one launch with the streams split over waves (bwd_split.hip).
struct BwdSplitArgs {
  View q, k, v, dout;
  const float* lse;
  const float* delta;
  MutView dq, dk, dv;
  Shape p;
  float* part;  // nsplit > 1: [split][dK, dV][B * Hkv * Skv][D] fp32
  int nsplit;   // workgroups per KV item
  int nw;       // waves per workgroup (4 or 8; D = 128: 4)
  int nkt;      // 32-row KV tiles (set by the launcher)
  int nrt;      // 32-row tiles of packed query rows per (b, hkv) (set by the launcher)
};

typedef hipError_t (*FwdLauncher)(const FwdArgs&, hipStream_t);
typedef hipError_t (*DecodeLauncher)(const DecodeArgs&, hipStream_t);
typedef hipError_t (*BwdLauncher)(const BwdArgs&, hipStream_t);
typedef hipError_t (*BwdSplitLauncher)(const BwdSplitArgs&, hipStream_t);

#define FLEXATT_DECL_D(D)                                                     \
  hipError_t fwd_mfma_bf16_d##D(const FwdArgs&, hipStream_t);                 \
  hipError_t fwd_mfma_f16_d##D(const FwdArgs&, hipStream_t);                  \
  hipError_t bwd_dq_mfma_bf16_d##D(const BwdArgs&, hipStream_t);              \
  hipError_t bwd_dq_mfma_f16_d##D(const BwdArgs&, hipStream_t);               \
  hipError_t bwd_dkdv_mfma_bf16_d##D(const BwdArgs&, hipStream_t);            \
  hipError_t bwd_dkdv_mfma_f16_d##D(const BwdArgs&, hipStream_t);

FLEXATT_DECL_D(32)
FLEXATT_DECL_D(64)
FLEXATT_DECL_D(128)
FLEXATT_DECL_D(256)
#undef FLEXATT_DECL_D
// D = 256 forward with wave-specialised pairs (fwd_ws.hip), called by the
// D = 256 forward launcher
hipError_t fwd_ws_bf16_d256(const FwdArgs&, hipStream_t);
hipError_t fwd_ws_f16_d256(const FwdArgs&, hipStream_t);
bool fwd_ws_fits(const Shape& p);  // its LDS (with a block map's lists) fits one CU

// [lo, hi) of every position's document (doc_bounds.hip): ids [B][S] integers
// of ids_bytes bytes, bounds int32 [B][S][2].
hipError_t doc_bounds_run(const void* ids, int ids_bytes, int B, int S, int* bounds, hipStream_t);

hipError_t bwd_delta(int dtype, const DeltaArgs&, hipStream_t);

// Split-KV forward (fwd_split.hip).
hipError_t fwd_split_bf16_d32(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_f16_d32(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_bf16_d64(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_f16_d64(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_bf16_d128(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_f16_d128(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_bf16_d256(const DecodeArgs&, hipStream_t);
hipError_t fwd_split_f16_d256(const DecodeArgs&, hipStream_t);

// Backward in one launch (bwd_split.hip), D <= 128.
hipError_t bwd_split_bf16_d32(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_f16_d32(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_bf16_d64(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_f16_d64(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_bf16_d128(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_f16_d128(const BwdSplitArgs&, hipStream_t);

// dK and dV from the splits' sums (a.part, a.nsplit), every D.
hipError_t bwd_split_sum_bf16_d32(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_f16_d32(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_bf16_d64(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_f16_d64(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_bf16_d128(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_f16_d128(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_bf16_d256(const BwdSplitArgs&, hipStream_t);
hipError_t bwd_split_sum_f16_d256(const BwdSplitArgs&, hipStream_t);

// The same two for fp32 inputs (f32_split.hip; the forward with one split), D <= 128.
hipError_t fwd_split_f32_d32(const DecodeArgs&, hipStream_t);
hipError_t bwd_split_f32_d32(const BwdSplitArgs&, hipStream_t);
hipError_t fwd_split_f32_d64(const DecodeArgs&, hipStream_t);
hipError_t bwd_split_f32_d64(const BwdSplitArgs&, hipStream_t);
hipError_t fwd_split_f32_d128(const DecodeArgs&, hipStream_t);
hipError_t bwd_split_f32_d128(const BwdSplitArgs&, hipStream_t);

// dK/dV as a KV-stationary tile stream (bwd_kv.hip), D = 64, 128 and 256.
hipError_t bwd_kv_bf16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_f16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_bf16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_f16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_bf16_d256(const BwdArgs&, hipStream_t);  // dV and dK passes as items of one launch
hipError_t bwd_kv_f16_d256(const BwdArgs&, hipStream_t);

// dK/dV that also writes its dS to a.ds (bwd_kv.hip), and dQ = scale * dS K
// from it (bwd_dq_ds.hip), D = 64, 128 and 256.
hipError_t bwd_kv_ds_bf16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_bf16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_bf16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_bf16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_bf16_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f16_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_bf16_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f16_d256(const BwdArgs&, hipStream_t);

// fp32 inputs on the fp32 matrix cores (f32_mfma.hip): forward, dK/dV (with
// or without writing dS), dQ from the staged dS and dQ recomputing S and dP,
// every D.
hipError_t fwd_f32_d32(const FwdArgs&, hipStream_t);
hipError_t fwd_f32_d64(const FwdArgs&, hipStream_t);
hipError_t fwd_f32_d128(const FwdArgs&, hipStream_t);
hipError_t fwd_f32_d256(const FwdArgs&, hipStream_t);
hipError_t bwd_dq_f32_d32(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_f32_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_f32_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_f32_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_dkdv_f32_d32(const BwdArgs&, hipStream_t);
hipError_t bwd_dkdv_f32_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_dkdv_f32_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_dkdv_f32_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f32_d32(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f32_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f32_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_kv_ds_f32_d256(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f32_d32(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f32_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f32_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_dq_ds_f32_d256(const BwdArgs&, hipStream_t);

// dQ as a query-stationary tile stream (bwd_q.hip), D = 64 and 128; with
// a.delta_out set it also computes Delta (written there) from O and dO.
hipError_t bwd_q_bf16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_q_f16_d128(const BwdArgs&, hipStream_t);
hipError_t bwd_q_bf16_d64(const BwdArgs&, hipStream_t);
hipError_t bwd_q_f16_d64(const BwdArgs&, hipStream_t);

}  // namespace flexatt
