// The float32-arithmetic backward of the scan (chunk_bwd_f32.hip), called by
// grm_hip_chunk_update_bwd for what the 16-bit MFMA kernels do not take.
#pragma once

#include <stdint.h>

#include <hip/hip_runtime.h>

namespace grmhip {

constexpr int BCT = 64;  // tokens per chunk (chunk_states granularity)

struct BwdGenArgs {
  const void* dh;
  const void* dmo;      // grad_memory_out
  const void* keys;
  const void* values;
  const void* queries;
  const void* memory;   // initial state
  const float* states;  // [B, n_chunks, dv, dk] state after each chunk
  float* gbuf;          // [B, n_chunks, dv, dk] slot ch: the adjoint at chunk ch's start (n_chunks > 1)
  float* part_k;        // [B, splits, T, dk] (splits > 1)
  float* part_q;        // [B, splits, T, dk]
  void* dq_out;
  void* dk_out;
  void* dv_out;
  void* dm_out;         // grad_memory, or float32 scratch that is copied there at the end
  int64_t batch;
  int64_t T;
  int dk;
  int dv;
  int n_chunks;
  int splits;           // workgroups sharing one chunk's value tiles
  int tiles_per_split;
  int mem_f32;
  int dm_f32;           // dm_out is float32
  int exact;            // infinities and NaN kept to the gradients that depend on them
  int vec_k;            // dk and the gradient rows allow 4-element stores
  int vec_v;            // dv likewise
  float c;
  float pw[BCT + 1];    // decay^0 .. decay^64
};

// Value columns per tile; the splits of a chunk are whole tiles.
constexpr int kGenDv = 32;

// Fills a.splits, tiles_per_split and the workspace pointers for the float32
// workspace of `floats` elements at ws, then launches.  key_dim <= 256 for
// 16-bit inputs, <= 128 for float32.
int launch_bwd_gen(BwdGenArgs a, int in_dtype, float* ws, int64_t floats, hipStream_t s);

}  // namespace grmhip
