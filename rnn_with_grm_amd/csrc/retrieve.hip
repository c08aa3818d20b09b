// Gather + query application over archived segment states, without
// materialising the gathered states, gfx950.
//
//   out[b, q, r, h] = sum_k memories[b, idx[b, q, r], h, k] * q'[b, q, k]
//
// which is the reference's apply_query_forward(batched_memory_gather(M, idx), q)
// (grm/core/cuda_ops.py:370-402; apply_query.cu:14-75 and batched_gather.cu:14-77
// for the two kernels it chains, paper_grm.py:229,301-313 for the composition),
// with q' = q cast to the memories' dtype as the caller does (paper_grm.py:301).
//
// The reference materialises [B, Q, R, d_v, d_k] (64 GiB at BASELINE config 3)
// and reads it back.  Here the (q, r) pairs of each sequence are first sorted by
// segment (one workgroup per sequence: LDS histogram, exclusive scan, scatter);
// then one workgroup per (sequence, segment, 128-row value tile) reads that
// archived state once into LDS and applies it to every query that selected it
// with fp32 MFMA (16x16x4), 64 pairs at a time.  Each pair's output row is
// written whole by exactly one workgroup, so the result does not depend on the
// order in which the sort placed pairs.
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "grm_hip.h"
#include "grm_hip_common.h"
#include "retrieve.h"

namespace grmhip {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int BK_THREADS = 1024;     // bucket kernels
constexpr int BK_ITEMS = 16384;      // pairs per workgroup when one sequence's pairs are split
constexpr int64_t kMultiBucketPairs = 4 * BK_ITEMS;  // from this many pairs per sequence
constexpr int64_t kMaxSegments = 16384;
constexpr int AP_THREADS = 256;      // apply kernel: 4 waves
constexpr int AP_V = kScaledTile;    // value rows per workgroup
constexpr int AP_N = 64;             // (q, r) pairs per tile

struct RetrieveArgs {
  const void* mem;
  const int64_t* idx;
  const void* queries;
  void* out;
  int32_t* offsets;  // [batch, segments + 1]
  int32_t* list;     // [batch, n_index]
  int32_t* bad;
  int64_t batch;
  int64_t segments;
  int64_t n_query;
  int64_t routes;
  int64_t n_index;  // n_query * routes
  int dv;
  int dk;
  int v_tiles;
  int32_t* partial;  // [batch, bk_chunks, segments]: per-chunk counts, then bases (multi-workgroup bucketing)
  int bk_chunks;     // pair groups of about BK_ITEMS per sequence (strided blocks of BK_THREADS pairs)
  // Work tiles of the apply kernels: at most tile_pairs consecutive pairs of
  // one segment each, so a segment that many queries selected is spread over
  // several workgroups.  tiles [batch, tb_max] of (segment, first pair, end, 0);
  // n_tiles [batch]; tile_base [batch, segments + 1] is the scan's scratch.
  int4* tiles;
  int32_t* n_tiles;
  int32_t* tile_base;
  int tb_max;
  int tile_pairs;
  // Gate-weighted, row-scaled 16-bit output (retrieve_fuse): out holds float16
  // rows of g * M q scaled by 2^sh per (pair, 128-value tile), scales[pair, tile] =
  // 2^-sh, 0 for a pair without a row.  nullptr: the plain [pairs, dv] output of
  // gather_apply.
  const float* gates;  // [batch, n_index]
  float* scales;       // [batch, n_index, v_tiles]
  int lds_rows;  // apply_lds_kernel makes the scaled rows
  int out_row;         // elements per output row (dv; dk for the queries' gradient)
};

// The query of pair `pid` (n_index <= INT32_MAX, so 32-bit unsigned division; -1
// stays -1).  The 64-bit quotient of an int by the int64_t route count was a
// branchy sequence of about 75 instructions in front of every query load:
// 16 x 65536 queries, 16 of 512 states, took 4.7 ms with it.
__device__ __forceinline__ int query_of(const RetrieveArgs& a, int pid) {
  return pid < 0 ? -1 : static_cast<int>(static_cast<uint32_t>(pid) / static_cast<uint32_t>(a.routes));
}

// ---------------------------------------------------------------------------
// Exclusive scan of hist[0..S) in LDS, in place, by one workgroup of
// BK_THREADS; offsets[s] gets the same values and offsets[S] the total.
__device__ void bucket_offsets(int* hist, int64_t S, int32_t* offsets) {
  __shared__ int wave_sum[BK_THREADS / 64];
  const int tid = threadIdx.x;
  // thread t owns bins [t per, (t + 1) per)
  const int per = static_cast<int>((S + BK_THREADS - 1) / BK_THREADS);
  const int lo = min(static_cast<int64_t>(tid) * per, S);
  const int hi = min(static_cast<int64_t>(lo) + per, S);
  int local = 0;
  for (int s = lo; s < hi; ++s) local += hist[s];
  const int lane = tid & 63, wave = tid >> 6;
  int incl = local;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wave; ++w) base += wave_sum[w];
  if (tid == 0) {
    int t = 0;
    for (int w = 0; w < BK_THREADS / 64; ++w) t += wave_sum[w];
    offsets[S] = t;
  }
  int run = base + incl - local;
  for (int s = lo; s < hi; ++s) {
    const int c = hist[s];
    offsets[s] = run;
    hist[s] = run;
    run += c;
  }
  __syncthreads();
}

// Lane index of the r-th set bit of mask (r < popcount(mask)).
__device__ __forceinline__ int nth_set_bit(uint64_t mask, int r) {
  int pos = 0;
#pragma unroll
  for (int w = 32; w >= 1; w >>= 1) {
    const int c = __popcll(mask & ((1ull << w) - 1u));
    if (r >= c) {
      r -= c;
      mask >>= w;
      pos += w;
    }
  }
  return pos;
}

// A row whose index is outside [0, segments): zeros, and one count.  Called
// by every lane of a wave together (bad: this lane's pair i is invalid).  Scaled
// rows only get the scale 0, which fuse_scaled_kernel takes as an absent row.
// With 16-byte rows the wave writes several whole rows per store instruction,
// coalesced (the first segments' short windows can leave most of a pair chunk
// empty); otherwise one row after another, consecutive lanes on consecutive
// elements.
template <class EM>
__device__ __forceinline__ void zero_rows_wave(const RetrieveArgs& a, int64_t b, int64_t i, bool bad) {
  using raw = typename ET<EM>::raw;
  uint64_t mask = __ballot(bad);
  const int lane = threadIdx.x & 63;
  if (mask != 0u && lane == 0 && a.bad != nullptr) atomicAdd(a.bad, static_cast<int>(__popcll(mask)));
  if (mask == 0u) return;
  if (a.scales != nullptr) {
    if (bad)
      for (int t = 0; t < a.v_tiles; ++t) a.scales[(b * a.n_index + i) * a.v_tiles + t] = 0.f;
    return;
  }
  const int64_t row_bytes = static_cast<int64_t>(a.out_row) * sizeof(raw);
  if (row_bytes % 16 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0) {
    // Whole rows in 16-byte pieces: lpr lanes per row, 64 / lpr rows per store
    // instruction, the rows taken in ballot order (i < n_index <= INT32_MAX).
    const int pieces = static_cast<int>(row_bytes / 16);
    int lpr = 1;
    while (lpr < pieces && lpr < 64) lpr <<= 1;
    const int m = __popcll(mask);
    const int i32 = static_cast<int>(i);
    for (int r0 = 0; r0 < m; r0 += 64 / lpr) {
      const int r = r0 + lane / lpr;
      const int row = __shfl(i32, nth_set_bit(mask, r < m ? r : 0), 64);
      if (r < m) {
        uint4* ob = reinterpret_cast<uint4*>(static_cast<raw*>(a.out) + (b * a.n_index + row) * a.out_row);
        for (int p = lane % lpr; p < pieces; p += lpr) ob[p] = uint4{0u, 0u, 0u, 0u};
      }
    }
    return;
  }
  while (mask != 0u) {
    const int l = __ffsll(static_cast<unsigned long long>(mask)) - 1;
    mask &= mask - 1u;
    const int64_t row = __shfl(i, l, 64);
    typename ET<EM>::raw* ob = static_cast<typename ET<EM>::raw*>(a.out) + (b * a.n_index + row) * a.out_row;
    for (int h = lane; h < a.out_row; h += 64) ob[h] = ET<EM>::from_f(0.f);
  }
}

// Pairs of one sequence sorted by segment, one workgroup per sequence.  Rows
// with an invalid index are zeroed here and never enter a bucket.
template <class EM>
__global__ __launch_bounds__(BK_THREADS) void bucket_kernel(const RetrieveArgs a) {
  extern __shared__ int hist[];  // [segments]
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.x;
  const int64_t S = a.segments, n = a.n_index;
  const int64_t* ib = a.idx + b * n;
  for (int64_t s = tid; s < S; s += BK_THREADS) hist[s] = 0;
  __syncthreads();
  for (int64_t i = tid; i < n; i += BK_THREADS) {
    const int64_t s = ib[i];
    if (s >= 0 && s < S) atomicAdd(&hist[s], 1);
  }
  __syncthreads();
  bucket_offsets(hist, S, a.offsets + b * (S + 1));
  int32_t* lb = a.list + b * n;
  for (int64_t i0 = 0; i0 < n; i0 += BK_THREADS) {  // uniform trip count: whole waves zero rows
    const int64_t i = i0 + tid;
    const int64_t s = i < n ? ib[i] : 0;
    const bool valid = s >= 0 && s < S;
    if (i < n && valid) lb[atomicAdd(&hist[s], 1)] = static_cast<int32_t>(i);
    zero_rows_wave<EM>(a, b, i, i < n && !valid);
  }
}

// The same sort over many workgroups per sequence (three launches): counts per
// pair group, per-(group, segment) bases, then the scatter.  The order of pairs
// inside a segment does not change any result, but it decides which query rows
// are read together.
// Scaled rows: group c holds consecutive blocks of BK_THREADS pairs, so that a
// segment's list follows the queries (in steps of a group) and workgroups on
// different segments sweep them together (16 x 65536 queries over 512 states, 16
// routes each: 3.60 -> 3.49 ms).
// Plain rows: group c holds the blocks c, c + bk_chunks, c + 2 bk_chunks, ...:
// the empty slots of the first segments' short windows, which can fill most of
// the first 16384 pairs, are then zeroed by every group instead of one or two.
struct PairBlocks {
  int64_t first, end, step;
  __device__ PairBlocks(const RetrieveArgs& a, int64_t group, int64_t n_blocks) {
    if (a.scales != nullptr) {
      const int64_t per = (n_blocks + a.bk_chunks - 1) / a.bk_chunks;
      first = group * per;
      end = min_i64(first + per, n_blocks);
      step = 1;
    } else {
      first = group;
      end = n_blocks;
      step = a.bk_chunks;
    }
  }
};

template <class EM>
__global__ __launch_bounds__(BK_THREADS) void bucket_count_kernel(const RetrieveArgs a) {
  extern __shared__ int hist[];  // [segments]
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.y, chunk = blockIdx.x;
  const int64_t S = a.segments, n = a.n_index;
  const int64_t n_blocks = (n + BK_THREADS - 1) / BK_THREADS;
  const int64_t* ib = a.idx + b * n;
  for (int64_t s = tid; s < S; s += BK_THREADS) hist[s] = 0;
  __syncthreads();
  const PairBlocks pb(a, chunk, n_blocks);
  for (int64_t blk = pb.first; blk < pb.end; blk += pb.step) {  // uniform trip count: whole waves zero rows
    const int64_t i = blk * BK_THREADS + tid;
    const int64_t s = i < n ? ib[i] : 0;
    const bool valid = s >= 0 && s < S;
    if (i < n && valid) atomicAdd(&hist[s], 1);
    zero_rows_wave<EM>(a, b, i, i < n && !valid);
  }
  __syncthreads();
  int32_t* pc = a.partial + (b * a.bk_chunks + chunk) * S;
  for (int64_t s = tid; s < S; s += BK_THREADS) pc[s] = hist[s];
}

__global__ __launch_bounds__(BK_THREADS) void bucket_bases_kernel(const RetrieveArgs a) {
  extern __shared__ int hist[];  // [segments]: totals, then segment offsets
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.x;
  const int64_t S = a.segments;
  int32_t* pb = a.partial + b * a.bk_chunks * S;
  for (int64_t s = tid; s < S; s += BK_THREADS) {
    int run = 0;
    for (int c = 0; c < a.bk_chunks; ++c) {
      const int v = pb[c * S + s];
      pb[c * S + s] = run;
      run += v;
    }
    hist[s] = run;
  }
  __syncthreads();
  bucket_offsets(hist, S, a.offsets + b * (S + 1));
  for (int64_t s = tid; s < S; s += BK_THREADS) {
    const int off = hist[s];
    for (int c = 0; c < a.bk_chunks; ++c) pb[c * S + s] += off;
  }
}

__global__ __launch_bounds__(BK_THREADS) void bucket_scatter_kernel(const RetrieveArgs a) {
  extern __shared__ int cur[];  // [segments]: next slot of each segment for this chunk
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.y, chunk = blockIdx.x;
  const int64_t S = a.segments, n = a.n_index;
  const int64_t n_blocks = (n + BK_THREADS - 1) / BK_THREADS;
  const int64_t* ib = a.idx + b * n;
  const int32_t* pc = a.partial + (b * a.bk_chunks + chunk) * S;
  for (int64_t s = tid; s < S; s += BK_THREADS) cur[s] = pc[s];
  __syncthreads();
  int32_t* lb = a.list + b * n;
  const PairBlocks pb(a, chunk, n_blocks);
  for (int64_t blk = pb.first; blk < pb.end; blk += pb.step) {  // the count kernel's pair group
    const int64_t i = blk * BK_THREADS + tid;
    if (i >= n) continue;
    const int64_t s = ib[i];
    if (s >= 0 && s < S) lb[atomicAdd(&cur[s], 1)] = static_cast<int32_t>(i);
  }
}

// The apply kernels' work list of one sequence: segment s with c pairs gives
// ceil(c / tile_pairs) tiles, in segment order (one workgroup per sequence).
__global__ __launch_bounds__(BK_THREADS) void tile_list_kernel(const RetrieveArgs a) {
  extern __shared__ int hist[];  // [segments]: tiles per segment, then their first slot
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.x;
  const int64_t S = a.segments;
  const int32_t* off = a.offsets + b * (S + 1);
  const int tp = a.tile_pairs;
  for (int64_t s = tid; s < S; s += BK_THREADS)
    hist[s] = static_cast<int>((static_cast<uint32_t>(off[s + 1] - off[s]) + tp - 1u) / static_cast<uint32_t>(tp));
  __syncthreads();
  int32_t* base = a.tile_base + b * (S + 1);
  bucket_offsets(hist, S, base);
  int4* tl = a.tiles + b * a.tb_max;
  for (int64_t s = tid; s < S; s += BK_THREADS) {
    int p = off[s], slot = hist[s];
    for (int left = off[s + 1] - p; left > 0; left -= tp) {
      const int take = min(left, tp);
      tl[slot++] = make_int4(static_cast<int>(s), p, p + take, 0);
      p += take;
    }
  }
  if (tid == 0) a.n_tiles[b] = base[S];
}

// Sixteen bytes of a row-major tile as fp32 values (8 elements for 16-bit types,
// 4 for float32); an OOB offset reads zeros.
template <class E>
__device__ __forceinline__ void load16_f32(__amdgpu_buffer_rsrc_t r, int off, float* dst) {
  const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  if constexpr (sizeof(typename ET<E>::raw) == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dst[2 * i] = ET<E>::to_f(static_cast<typename ET<E>::raw>(u[i] & 0xffffu));
      dst[2 * i + 1] = ET<E>::to_f(static_cast<typename ET<E>::raw>(u[i] >> 16));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = __uint_as_float(u[i]);
  }
}

// ---------------------------------------------------------------------------
// One workgroup per (sequence, segment, 128-row value tile).  Wave w computes
// value rows [32w, 32w + 32) for 64 pairs: D[v][p] = sum_k M[v][k] q'[p][k]
// with A = state rows v, B = query rows p (lane (g, n) of a 16x16x4 operand
// holds row n, key 4kk + g).
template <class EL, class EM, class EQ, int DKP, bool VEC>
__global__ __launch_bounds__(AP_THREADS) void apply_bucket_kernel(const RetrieveArgs a) {
  using rawl = typename ET<EL>::raw;  // stored memories
  using rawm = typename ET<EM>::raw;  // arithmetic / output type
  using rawq = typename ET<EQ>::raw;
  constexpr int MS = DKP + 4;                            // state tile row stride (floats)
  constexpr int QS = (DKP > AP_V ? DKP : AP_V) + 4;      // query / output tile row stride
  constexpr int EPU_M = 16 / sizeof(rawl);               // elements per 16-byte unit
  constexpr int EPU_Q = 16 / sizeof(rawq);
  constexpr int UPR_M = DKP / EPU_M;                     // units per padded row
  constexpr int UPR_Q = DKP / EPU_Q;
  constexpr int M_UNITS = AP_V * UPR_M / AP_THREADS;     // per thread
  constexpr int Q_UNITS = (AP_N * UPR_Q + AP_THREADS - 1) / AP_THREADS;
  static_assert(M_UNITS * AP_THREADS == AP_V * UPR_M, "state tile splits evenly");
  extern __shared__ __align__(16) float sm[];
  float* Ms = sm;              // [AP_V][MS]
  float* QO = Ms + AP_V * MS;  // [AP_N][QS]: queries, then the output tile
  __shared__ int pair_id[AP_N];

  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t vt = blockIdx.x % a.v_tiles;
  const int64_t tile = blockIdx.x / a.v_tiles;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int64_t s = te.x;
  const int p_begin = te.y, p_end = te.z;
  const int dk = a.dk, dv = a.dv;
  const int v0 = static_cast<int>(vt) * AP_V;

  // State rows v0 .. v0 + 127 as fp32, zero past d_v and d_k.
  const rawl* msrc = static_cast<const rawl*>(a.mem) + (b * a.segments + s) * dv * dk;
  if constexpr (VEC) {
    const __amdgpu_buffer_rsrc_t rm = make_rsrc(msrc, static_cast<uint32_t>(dv * dk * sizeof(rawl)));
    float x[M_UNITS][EPU_M];
#pragma unroll
    for (int u = 0; u < M_UNITS; ++u) {
      const int e = tid + AP_THREADS * u;
      const int v = e / UPR_M, c = (e % UPR_M) * EPU_M;
      load16_f32<EL>(rm, (v0 + v < dv && c < dk) ? ((v0 + v) * dk + c) * static_cast<int>(sizeof(rawl)) : kBufOOB,
                     x[u]);
    }
#pragma unroll
    for (int u = 0; u < M_UNITS; ++u) {
      const int e = tid + AP_THREADS * u;
      const int v = e / UPR_M, c = (e % UPR_M) * EPU_M;
#pragma unroll
      for (int i = 0; i < EPU_M; i += 4)
        *reinterpret_cast<f32x4*>(Ms + v * MS + c + i) = f32x4{x[u][i], x[u][i + 1], x[u][i + 2], x[u][i + 3]};
    }
  } else {
    for (int e = tid; e < AP_V * DKP; e += AP_THREADS) {
      const int v = e / DKP, k = e % DKP;
      Ms[v * MS + k] = (v0 + v < dv && k < dk) ? ET<EL>::to_f(msrc[(v0 + v) * dk + k]) : 0.f;
    }
  }
  const int32_t* lb = a.list + b * a.n_index;
  const rawq* qsrc = static_cast<const rawq*>(a.queries) + b * a.n_query * dk;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(qsrc, static_cast<uint32_t>(a.n_query * dk * sizeof(rawq)));
  rawm* obase = static_cast<rawm*>(a.out) + b * a.n_index * dv;

  for (int p0 = p_begin; p0 < p_end; p0 += AP_N) {
    const int np = min(AP_N, p_end - p0);
    __syncthreads();  // state tile in place; previous output tile written out
    if (tid < AP_N) pair_id[tid] = tid < np ? lb[p0 + tid] : -1;
    __syncthreads();
    // Query rows of the tile's pairs, cast to the memories' dtype (the caller's
    // cast of q), as fp32.
    if constexpr (VEC) {
      float x[Q_UNITS][EPU_Q];
#pragma unroll
      for (int u = 0; u < Q_UNITS; ++u) {
        const int e = tid + AP_THREADS * u;
        const int p = min(e / UPR_Q, AP_N - 1), c = (e % UPR_Q) * EPU_Q;
        const int pid = pair_id[p];
        const int qoff = (e < AP_N * UPR_Q && pid >= 0 && c < dk)
                             ? (query_of(a, pid) * dk + c) * static_cast<int>(sizeof(rawq))
                             : kBufOOB;
        load16_f32<EQ>(rq, qoff, x[u]);
      }
#pragma unroll
      for (int u = 0; u < Q_UNITS; ++u) {
        const int e = tid + AP_THREADS * u;
        if (e >= AP_N * UPR_Q) continue;
        const int p = e / UPR_Q, c = (e % UPR_Q) * EPU_Q;
#pragma unroll
        for (int i = 0; i < EPU_Q; i += 4) {
          f32x4 y;
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = ET<EM>::to_f(ET<EM>::from_f(x[u][i + j]));
          *reinterpret_cast<f32x4*>(QO + p * QS + c + i) = y;
        }
      }
    } else {
      for (int e = tid; e < AP_N * DKP; e += AP_THREADS) {
        const int p = e / DKP, k = e % DKP;
        const int pid = pair_id[p];
        float x = 0.f;
        if (pid >= 0 && k < dk) {
          const rawq q = qsrc[static_cast<int64_t>(query_of(a, pid)) * dk + k];
          x = ET<EM>::to_f(ET<EM>::from_f(ET<EQ>::to_f(q)));
        }
        QO[p * QS + k] = x;
      }
    }
    __syncthreads();
    f32x4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int kk = 0; kk < DKP / 4; ++kk) {
      float av[2], bv[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) av[i] = Ms[(32 * w + 16 * i + n) * MS + 4 * kk + g];
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[j] = QO[(16 * j + n) * QS + 4 * kk + g];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();  // query tile consumed
    // lane (g, n) holds D[v = 32w + 16i + 4g + r][p = 16j + n]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(QO + (16 * j + n) * QS + 32 * w + 16 * i + 4 * g) = acc[i][j];
    __syncthreads();
    // whole output rows: pair p -> out[b, pair_id[p], v0 .. v0 + 127]
    const int vcols = min(AP_V, dv - v0);
    for (int e = tid; e < np * AP_V; e += AP_THREADS) {
      const int p = e / AP_V, v = e % AP_V;
      if (v < vcols) obase[static_cast<int64_t>(pair_id[p]) * dv + v0 + v] = ET<EM>::from_f(QO[p * QS + v]);
    }
  }
}

// Register-operand variant (16-byte aligned rows): no input tiles in LDS.  The
// key order of every 4-deep fp32 MFMA step is permuted so that lane group g
// owns keys [g*KG, (g+1)*KG), KG = DKP / 4: step t uses key g*KG + t in group g.
// A lane then holds 32 (for d_k = 128) consecutive keys of its state row and of
// its pair's query row, both loaded with 16-byte vector loads straight into the
// operand registers.  Only the output tile goes through LDS (for whole-row
// stores), so two or three workgroups share a CU and hide each other's latency.
template <class EL, class EM, class EQ, int DKP>
__global__ __launch_bounds__(AP_THREADS) void apply_reg_kernel(const RetrieveArgs a) {
  using rawl = typename ET<EL>::raw;  // stored memories
  using rawm = typename ET<EM>::raw;  // arithmetic / output type
  using rawq = typename ET<EQ>::raw;
  constexpr int KG = DKP / 4;                       // keys per lane group
  constexpr int OS = AP_V + 4;                      // output tile row stride (floats)
  constexpr int EPU_M = 16 / sizeof(rawl);
  constexpr int EPU_Q = 16 / sizeof(rawq);
  static_assert(KG % EPU_M == 0 && KG % EPU_Q == 0, "a lane's keys are whole 16-byte units");
  __shared__ __align__(16) float Os[AP_N * OS];

  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t vt = blockIdx.x % a.v_tiles;
  const int64_t tile = blockIdx.x / a.v_tiles;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int64_t s = te.x;
  const int p_begin = te.y, p_end = te.z;
  const int dk = a.dk, dv = a.dv;
  const int v0 = static_cast<int>(vt) * AP_V;
  const int k0 = g * KG;

  // A operands: state rows v = v0 + 32w + 16i + n, keys k0 .. k0 + KG - 1.
  const rawl* msrc = static_cast<const rawl*>(a.mem) + (b * a.segments + s) * dv * dk;
  const __amdgpu_buffer_rsrc_t rm = make_rsrc(msrc, static_cast<uint32_t>(dv * dk * sizeof(rawl)));
  float am[2][KG];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = v0 + 32 * w + 16 * i + n;
#pragma unroll
    for (int u = 0; u < KG / EPU_M; ++u) {
      const int k = k0 + u * EPU_M;
      load16_f32<EL>(rm, (v < dv && k < dk) ? (v * dk + k) * static_cast<int>(sizeof(rawl)) : kBufOOB,
                     &am[i][u * EPU_M]);
    }
  }
  const int32_t* lb = a.list + b * a.n_index;
  const rawq* qsrc = static_cast<const rawq*>(a.queries) + b * a.n_query * dk;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(qsrc, static_cast<uint32_t>(a.n_query * dk * sizeof(rawq)));
  rawm* obase = static_cast<rawm*>(a.out) + b * a.n_index * dv;
  const int vcols = min(AP_V, dv - v0);

  for (int p0 = p_begin; p0 < p_end; p0 += AP_N) {
    const int np = min(AP_N, p_end - p0);
    f32x4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // B operand: the query of pair 16j + n, keys k0 .. k0 + KG - 1, cast to
      // the memories' dtype (the caller's cast of q).
      const int p = 16 * j + n;
      const int qrow = query_of(a, p < np ? lb[p0 + p] : -1);
      float bq[KG];
#pragma unroll
      for (int u = 0; u < KG / EPU_Q; ++u) {
        const int k = k0 + u * EPU_Q;
        load16_f32<EQ>(rq, (qrow >= 0 && k < dk) ? (qrow * dk + k) * static_cast<int>(sizeof(rawq)) : kBufOOB,
                       &bq[u * EPU_Q]);
      }
#pragma unroll
      for (int t = 0; t < KG; ++t) bq[t] = ET<EM>::to_f(ET<EM>::from_f(bq[t]));
#pragma unroll
      for (int t = 0; t < KG; ++t) {
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(am[i][t], bq[t], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();  // previous output tile written out
    // lane (g, n) holds D[v = 32w + 16i + 4g + r][p = 16j + n]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(Os + (16 * j + n) * OS + 32 * w + 16 * i + 4 * g) = acc[i][j];
    __syncthreads();
    // whole output rows, four values per thread: pair p -> out[b, pair, v0 .. v0 + 127]
    for (int e = tid; e < np * (AP_V / 4); e += AP_THREADS) {
      const int p = e / (AP_V / 4), v = (e % (AP_V / 4)) * 4;
      const int pid = lb[p0 + p];
      const f32x4 val = *reinterpret_cast<const f32x4*>(Os + p * OS + v);
      rawm* dst = obase + static_cast<int64_t>(pid) * dv + v0 + v;
      if (v + 4 <= vcols) {
        store4_raw<EM>(dst, val);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (v + r < vcols) dst[r] = ET<EM>::from_f(val[r]);
      }
    }
  }
}

// 16-bit MFMA variant, exact: the memories are split into NPART parts of the
// MFMA input type EF (one part when EM is EF; hi + mid + lo bf16 parts, which
// together hold all 24 mantissa bits, when EM is float32), and the query cast
// to EM is exact in EF, so every product is exact and only the float32
// accumulation rounds, as in a float32 dot product.  MFMA step c (16x16x32)
// takes keys 32c + 8g .. + 7 from lane group g, so the four groups of a row
// read consecutive bytes: each state load instruction covers whole 128-byte
// lines of 16 rows (fp32 states) instead of 16-byte pieces of 64 lines.
// A step of up to 32 pairs leaves out the products and stores of its upper half:
// with about 64 pairs per state every other state ends on a step of a few (64 x 2048
// queries, 8 of 256 states of 128 x 128: 461 -> 455 us for the whole call; tested
// every 16 pairs, 460 us).
template <class EL, class EM, class EQ, int DKP, class EF, int NPART, bool SCALED = false>
__global__ __launch_bounds__(AP_THREADS) void apply_mfma16_kernel(const RetrieveArgs a) {
  using rawl = typename ET<EL>::raw;  // stored memories
  using rawm = typename ET<EM>::raw;  // arithmetic / output type
  using rawq = typename ET<EQ>::raw;
  constexpr int KG = DKP / 4;
  constexpr int NSTEP = KG / 8;
  constexpr int OS = AP_V + 4;
  constexpr int EPU_M = 16 / sizeof(rawl);
  constexpr int EPU_Q = 16 / sizeof(rawq);
  static_assert(KG % 8 == 0 && KG % EPU_M == 0 && KG % EPU_Q == 0, "a lane's keys are whole MFMA slots");
  static_assert(AP_N == 64, "one pair per lane");
  __shared__ __align__(16) float Os[AP_N * OS];

  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t vt = blockIdx.x % a.v_tiles;
  const int64_t tile = blockIdx.x / a.v_tiles;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int64_t s = te.x;
  const int p_begin = te.y, p_end = te.z;
  const int dk = a.dk, dv = a.dv;
  const int v0 = static_cast<int>(vt) * AP_V;
  // Register slot x (0 .. KG - 1) of a lane's state row / query holds key key_of(x).
  auto key_of = [&](int x) { return 32 * (x >> 3) + 8 * g + (x & 7); };
  static_assert(EPU_M <= 8 && EPU_Q <= 8, "a 16-byte load stays inside one MFMA slot group");
  const int32_t* lb = a.list + b * a.n_index;
  // Pair ids of the first tile, one per lane (issued before the state loads so
  // that waiting for them does not wait for the state).
  int pid_l = lane < p_end - p_begin ? lb[p_begin + lane] : -1;

  const rawl* msrc = static_cast<const rawl*>(a.mem) + (b * a.segments + s) * dv * dk;
  const __amdgpu_buffer_rsrc_t rm = make_rsrc(msrc, static_cast<uint32_t>(dv * dk * sizeof(rawl)));
  float xm[2][KG];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = v0 + 32 * w + 16 * i + n;
#pragma unroll
    for (int u = 0; u < KG / EPU_M; ++u) {
      const int k = key_of(u * EPU_M);
      load16_f32<EL>(rm, (v < dv && k < dk) ? (v * dk + k) * static_cast<int>(sizeof(rawl)) : kBufOOB,
                     &xm[i][u * EPU_M]);
    }
  }
  const rawq* qsrc = static_cast<const rawq*>(a.queries) + b * a.n_query * dk;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(qsrc, static_cast<uint32_t>(a.n_query * dk * sizeof(rawq)));
  rawm* obase = static_cast<rawm*>(a.out) + b * a.n_index * dv;
  const int vcols = min(AP_V, dv - v0);

  Frag8<EF> am[2][NPART][NSTEP];
  bool split = false;
  // The query's MFMA operand: q cast to EM, then to EF.  When both casts are
  // exact (a 16-bit query of type EF, EM float32 or EF) the operand is the
  // query's own bits, loaded as they are (half the registers of float32).
  constexpr bool kRawQ = std::is_same_v<EQ, EF> && (std::is_same_v<EM, F32> || std::is_same_v<EM, EQ>);
  float xq[kRawQ ? 1 : 4][kRawQ ? 1 : KG];
  Frag8<EF> rq8[4][kRawQ ? NSTEP : 1];
  // Query rows of a 64-pair step: lane 16 j + n holds pair j's row in slot j.
  // The loads of step s + 1 are issued right after step s's products, so they
  // overlap its output tile instead of opening the next step.
  auto load_q = [&](int pid_src) {
    const int qrow_src = query_of(a, pid_src);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int qrow = __shfl(qrow_src, 16 * j + n, 64);
      if constexpr (kRawQ) {
#pragma unroll
        for (int c = 0; c < NSTEP; ++c) {
          const int k = key_of(8 * c);
          const int off = (qrow >= 0 && k < dk) ? (qrow * dk + k) * static_cast<int>(sizeof(rawq)) : kBufOOB;
          rq8[j][c] = __builtin_bit_cast(Frag8<EF>, __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0));
        }
      } else {
#pragma unroll
        for (int u = 0; u < KG / EPU_Q; ++u) {
          const int k = key_of(u * EPU_Q);
          load16_f32<EQ>(rq, (qrow >= 0 && k < dk) ? (qrow * dk + k) * static_cast<int>(sizeof(rawq)) : kBufOOB,
                         &xq[j][u * EPU_Q]);
        }
      }
    }
  };
  load_q(pid_l);
  for (int p0 = p_begin; p0 < p_end; p0 += AP_N) {
    const int np = __builtin_amdgcn_readfirstlane(min(AP_N, p_end - p0));
    const int pid_cur = pid_l;
    const bool more = p0 + AP_N < p_end;
    const int pid_next = (more && lane < p_end - p0 - AP_N) ? lb[p0 + AP_N + lane] : -1;
    // The gate of this lane's pair, loaded while the tile's products run.
    float gate_cur = 0.f;
    if constexpr (SCALED) gate_cur = pid_cur >= 0 ? a.gates[b * a.n_index + pid_cur] : 0.f;
    if (!split) {
      split = true;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < NSTEP; ++c)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float rest = xm[i][8 * c + e];
#pragma unroll
            for (int part = 0; part < NPART; ++part) {
              const typename ET<EF>::raw h = ET<EF>::from_f(rest);
              am[i][part][c].e[e] = h;
              rest -= ET<EF>::to_f(h);
            }
          }
    }
    f32x4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j == 2 && np <= 32) break;  // no pairs in the upper half
      Frag8<EF> bq[NSTEP];
#pragma unroll
      for (int c = 0; c < NSTEP; ++c) {
        if constexpr (kRawQ) {
          bq[c] = rq8[j][c];
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) bq[c].e[e] = ET<EF>::from_f(ET<EM>::to_f(ET<EM>::from_f(xq[j][8 * c + e])));
        }
      }
#pragma unroll
      for (int c = 0; c < NSTEP; ++c)
#pragma unroll
        for (int part = 0; part < NPART; ++part)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[i][j] = mfma8(am[i][part][c], bq[c], acc[i][j]);
    }
    if (more) load_q(pid_next);
    pid_l = pid_next;
    __syncthreads();  // previous output tile written out
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(Os + (16 * j + n) * OS + 32 * w + 16 * i + 4 * g) = acc[i][j];
    __syncthreads();
    constexpr int PER = AP_N * (AP_V / 4) / AP_THREADS;  // stores per thread per full tile
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      if (it == PER / 2 && np <= 32) break;
      const int e = tid + AP_THREADS * it;
      const int p = e / (AP_V / 4), v = (e % (AP_V / 4)) * 4;
      const int pid = __shfl(pid_cur, p, 64);
      if constexpr (SCALED) {
        // The 32 lanes of one half-wave hold pair p's 128 values of this tile:
        // scale the gate-weighted row so its largest magnitude lies in [2^14, 2^15)
        // and store it as float16 with the inverse power of two.
        const float gp = __shfl(gate_cur, p, 64);
        const f32x4 val = *reinterpret_cast<const f32x4*>(Os + p * OS + v) * gp;
        float m = fmaxf(fmaxf(fabsf(val[0]), fabsf(val[1])), fmaxf(fabsf(val[2]), fabsf(val[3])));
        // maximum over the 32 lanes of the half-wave without LDS: quad swaps, the
        // half-row and row mirrors (DPP), then the 16-lane row swap
        m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0xb1, 0xf, 0xf, false)));
        m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x4e, 0xf, 0xf, false)));
        m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x141, 0xf, 0xf, false)));
        m = fmaxf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x140, 0xf, 0xf, false)));
        {
          const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
          m = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        }
        int ex = 0;
        (void)frexpf(m, &ex);
        const int sh = min(max(15 - ex, -100), 100);
        if (p < np) {
          uint16_t* dst = static_cast<uint16_t*>(a.out) + (b * a.n_index + pid) * static_cast<int64_t>(dv) + v0 + v;
          if (v + 4 <= vcols) {
            uint2 q;
            q.x = pack2<F16>(ldexpf(val[0], sh), ldexpf(val[1], sh));
            q.y = pack2<F16>(ldexpf(val[2], sh), ldexpf(val[3], sh));
            *reinterpret_cast<uint2*>(dst) = q;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (v + r < vcols) dst[r] = ET<F16>::from_f(ldexpf(val[r], sh));
          }
          if ((tid & 31) == 0) a.scales[(b * a.n_index + pid) * a.v_tiles + vt] = ldexpf(1.f, -sh);
        }
        continue;
      }
      if (p < np) {
        const f32x4 val = *reinterpret_cast<const f32x4*>(Os + p * OS + v);
        rawm* dst = obase + static_cast<int64_t>(pid) * dv + v0 + v;
        if (v + 4 <= vcols) {
          store4_raw<EM>(dst, val);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (v + r < vcols) dst[r] = ET<EM>::from_f(val[r]);
        }
      }
    }
  }
}

template <class EL, class EM, class EQ, int DKP, class EF, int NPART, bool SCALED = false>
int launch_apply_mfma16(const RetrieveArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(a.tb_max) * a.v_tiles), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_mfma16_kernel<EL, EM, EQ, DKP, EF, NPART, SCALED>), grid,
                     dim3(AP_THREADS), 0, s, a);
  return check_launch("gather_apply");
}

template <class EL, class EM, class EQ, int DKP>
int launch_apply_reg(const RetrieveArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(a.tb_max) * a.v_tiles), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_reg_kernel<EL, EM, EQ, DKP>), grid, dim3(AP_THREADS), 0, s,
                     a);
  return check_launch("gather_apply");
}

template <class EL, class EM, class EQ, int DKP, bool VEC>
int launch_apply(const RetrieveArgs& a, hipStream_t s) {
  constexpr int MS = DKP + 4;
  constexpr int QS = (DKP > AP_V ? DKP : AP_V) + 4;
  constexpr size_t lds = (static_cast<size_t>(AP_V) * MS + static_cast<size_t>(AP_N) * QS) * sizeof(float);
  static_assert(lds <= 160 * 1024, "apply tiles fit one CU's LDS");
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&apply_bucket_kernel<EL, EM, EQ, DKP, VEC>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) {
      set_error("gather_apply: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
    attr_set = true;
  }
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(a.tb_max) * a.v_tiles), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_bucket_kernel<EL, EM, EQ, DKP, VEC>), grid,
                     dim3(AP_THREADS), lds, s, a);
  return check_launch("gather_apply");
}

// 16-byte tile loads need whole units per row and 16-byte aligned bases.
template <class EL, class EQ>
bool vec_ok(const RetrieveArgs& a) {
  const int el = 16 / static_cast<int>(sizeof(typename ET<EL>::raw));
  const int eq = 16 / static_cast<int>(sizeof(typename ET<EQ>::raw));
  return a.dk % el == 0 && a.dk % eq == 0 && reinterpret_cast<uintptr_t>(a.mem) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(a.queries) % 16 == 0 &&
         a.dv * static_cast<int64_t>(a.dk) * static_cast<int64_t>(sizeof(typename ET<EL>::raw)) < INT32_MAX &&
         a.n_query * static_cast<int64_t>(a.dk) * static_cast<int64_t>(sizeof(typename ET<EQ>::raw)) < INT32_MAX;
}

template <class EL, class EM, class EQ>
int dispatch_dk(const RetrieveArgs& a, hipStream_t s) {
  if (vec_ok<EL, EQ>(a)) {
    using Plan = MfmaPlan<EL, EM, EQ>;
    if constexpr (Plan::ok) {
      using EF = typename Plan::EF;
      constexpr int NPART = Plan::parts;
      if (a.dk <= 32) return launch_apply_mfma16<EL, EM, EQ, 32, EF, NPART>(a, s);
      if (a.dk <= 64) return launch_apply_mfma16<EL, EM, EQ, 64, EF, NPART>(a, s);
      return launch_apply_mfma16<EL, EM, EQ, 128, EF, NPART>(a, s);
    } else {
      if (a.dk <= 32) return launch_apply_reg<EL, EM, EQ, 32>(a, s);
      if (a.dk <= 64) return launch_apply_reg<EL, EM, EQ, 64>(a, s);
      return launch_apply_reg<EL, EM, EQ, 128>(a, s);
    }
  }
  if (a.dk <= 32) return launch_apply<EL, EM, EQ, 32, false>(a, s);
  if (a.dk <= 64) return launch_apply<EL, EM, EQ, 64, false>(a, s);
  return launch_apply<EL, EM, EQ, 128, false>(a, s);
}

template <class EL, class EM>
int dispatch_q(const RetrieveArgs& a, int q_dtype, hipStream_t s) {
  switch (q_dtype) {
    case GRM_HIP_F32: return dispatch_dk<EL, EM, F32>(a, s);
    case GRM_HIP_F16: return dispatch_dk<EL, EM, F16>(a, s);
    default: return dispatch_dk<EL, EM, BF16>(a, s);
  }
}

// ---------------------------------------------------------------------------
// Residual + LayerNorm over the scaled rows of retrieve_fuse:
//   out[t] = LN(h[t] + sum_r scales[t, r, c / 128] * rows[t, r, c])
// h and out in E, the LayerNorm weight and bias in float32,
// with r in order 0 .. R-1 (the gates are already in the rows; scale 0: no row), a
// two-pass mean / variance in fp32.  lpr lanes share a row, each covering NV groups of
// 8 consecutive columns (16-byte float16 loads of the rows).

template <class E>
__device__ __forceinline__ void load8(__amdgpu_buffer_rsrc_t r, int off, float (&f)[8]) {
  if constexpr (sizeof(typename ET<E>::raw) == 2) {
    const U8<E> u = __builtin_bit_cast(U8<E>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = ET<E>::to_f(u.e[e]);
  } else {
    const u32x4 lo = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    const u32x4 hi = __builtin_amdgcn_raw_buffer_load_b128(r, off == kBufOOB ? kBufOOB : off + 16, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = __uint_as_float(lo[e]);
      f[4 + e] = __uint_as_float(hi[e]);
    }
  }
}

template <class E>
__device__ __forceinline__ void store8(__amdgpu_buffer_rsrc_t r, int off, const float (&y)[8]) {
  if constexpr (sizeof(typename ET<E>::raw) == 2) {
    const u32x4 q = u32x4{pack2<E>(y[0], y[1]), pack2<E>(y[2], y[3]), pack2<E>(y[4], y[5]), pack2<E>(y[6], y[7])};
    __builtin_amdgcn_raw_buffer_store_b128(q, r, off, 0, 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b128(
        u32x4{__float_as_uint(y[0]), __float_as_uint(y[1]), __float_as_uint(y[2]), __float_as_uint(y[3])}, r, off, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(
        u32x4{__float_as_uint(y[4]), __float_as_uint(y[5]), __float_as_uint(y[6]), __float_as_uint(y[7])}, r,
        off == kBufOOB ? kBufOOB : off + 16, 0, 0);
  }
}

template <class E, int NV>
__global__ __launch_bounds__(256) void fuse_scaled_kernel(const FuseScaledArgs a, const int lpr) {
  using raw = typename ET<E>::raw;
  const int tid = threadIdx.x;
  const int sub = tid & (lpr - 1);
  const int lane = tid & 63, per = min(lpr, AP_V / 8);  // lanes on one tile of a row (or the row)
  const WaveRows wr = wave_rows(static_cast<int64_t>(blockIdx.x) * (256 / lpr), lpr, a.n_rows);
  const bool live = wr.row < a.n_rows;
  const int H = a.hidden;
  const int64_t rr = live ? wr.row : 0;
  const int hb = H * static_cast<int>(sizeof(raw)), rowb = a.routes * H * 2;  // row bytes of h / out, of rows
  const __amdgpu_buffer_rsrc_t rh = wave_rows_rsrc(a.h, wr, hb);
  const __amdgpu_buffer_rsrc_t rrow = wave_rows_rsrc(a.rows, wr, rowb);
  const float* sc = a.scales + rr * a.routes * a.v_tiles;
  float x[NV][8];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = (sub + lpr * v) * 8;
    const bool in = live && c < H;
    float hv[8];
    load8<E>(rh, in ? wr.local * hb + c * static_cast<int>(sizeof(raw)) : kBufOOB, hv);
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = 0.f;
    const int tile = c / AP_V;
    if (a.all_there != 0 && a.routes == 1) {  // the window retrieval's sums
      const float s0 = in ? sc[tile] : 0.f;
      float rv[8];
      load8<F16>(rrow, in ? wr.local * rowb + c * 2 : kBufOOB, rv);
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = fmaf(s0, rv[e], r[e]);
    } else
    // The scales of 16 routes at a time (fewer with short rows), one per lane of
    // the lanes on one tile; rows without a scale are not read.
    for (int j0 = 0; j0 < a.routes; j0 += per) {
      const int jl = j0 + (lane & (per - 1));
      const bool have = live && tile < a.v_tiles && jl < a.routes;  // also on lanes past the row's end
      const float sl = have ? sc[jl * a.v_tiles + tile] : 0.f;
      const uint64_t rows_there = __ballot(sl != 0.f);
#pragma unroll 4
      for (int t = 0; t < min(per, a.routes - j0); ++t) {
        const int src = (lane & ~(per - 1)) + t;
        const float sj = __shfl(sl, src, 64);
        float rv[8];
        load8<F16>(rrow, in && ((rows_there >> src) & 1) ? wr.local * rowb + ((j0 + t) * H + c) * 2 : kBufOOB, rv);
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = fmaf(sj, rv[e], r[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x[v][e] = c < H ? hv[e] + r[e] : 0.f;
  }
  const __amdgpu_buffer_rsrc_t ro = wave_rows_rsrc(a.out, wr, hb);
  auto out_off = [&](int v) {
    const int c = (sub + lpr * v) * 8;
    return (live && c < H) ? wr.local * hb + c * static_cast<int>(sizeof(raw)) : kBufOOB;
  };
  if (a.w == nullptr) {
#pragma unroll
    for (int v = 0; v < NV; ++v) store8<E>(ro, out_off(v), x[v]);
    return;
  }
  float sum = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 8; ++e) sum += x[v][e];
  for (int off = lpr >> 1; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  const float mean = sum / static_cast<float>(H);
  float var = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = (sub + lpr * v) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = x[v][e] - mean;
      var = c < H ? fmaf(d, d, var) : var;
    }
  }
  for (int off = lpr >> 1; off > 0; off >>= 1) var += __shfl_xor(var, off, 64);
  const float rstd = 1.0f / sqrtf(var / static_cast<float>(H) + a.eps);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w, H * 4);
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(a.bias, a.bias != nullptr ? H * 4 : 0u);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = (sub + lpr * v) * 8;
    const int off = c < H ? c * 4 : kBufOOB;
    float wv[8], bv[8];
    load8<F32>(rw, off, wv);  // LayerNorm parameters are float32
    load8<F32>(rb, off, bv);  // zeros without a bias
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (x[v][e] - mean) * rstd * wv[e] + bv[e];
    store8<E>(ro, out_off(v), y);
  }
}

template <class E>
int launch_fuse_scaled(const FuseScaledArgs& a, hipStream_t s) {
  const int groups = a.hidden / 8;
  int lpr = 1;
  while (lpr < 64 && lpr < groups) lpr <<= 1;
  const int nv = (groups + lpr - 1) / lpr;
  const dim3 grid(static_cast<unsigned>((a.n_rows + 256 / lpr - 1) / (256 / lpr)));
  auto go = [&](auto nvc) {
    hipLaunchKernelGGL((fuse_scaled_kernel<E, decltype(nvc)::value>), grid, dim3(256), 0, s, a, lpr);
  };
  if (nv <= 1) go(std::integral_constant<int, 1>{});
  else if (nv <= 2) go(std::integral_constant<int, 2>{});
  else if (nv <= 4) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 8>{});
  return check_launch("retrieve_fuse(fuse)");
}

}  // namespace

int fuse_scaled(const FuseScaledArgs& a, int h_dtype, hipStream_t s) {
  switch (h_dtype) {
    case GRM_HIP_F32: return launch_fuse_scaled<F32>(a, s);
    case GRM_HIP_F16: return launch_fuse_scaled<F16>(a, s);
    default: return launch_fuse_scaled<BF16>(a, s);
  }
}

namespace {

// Many pairs per state, for the scaled rows of retrieve_fuse: the state's MFMA
// operands in LDS, the pairs in registers.  Eight waves stage one 16 NI-row value
// tile of the segment's state as NPART exact 16-bit parts in fragment order (1 KB
// per fragment, read back without bank conflicts), then each wave takes 48 pairs
// at a time on its own, with no barrier: an A fragment read from LDS serves three
// MFMAs, and a lane ends with a quarter of each of three pairs' rows, so
// the gate, the row's scale and the 16-bit rows come straight from the
// accumulators.  Row m = 4 g' + r of fragment i stands for value 32 (i >> 1) + 8 g' +
// 4 (i & 1) + r: lane (g, n)'s accumulators of fragments 2p and 2p + 1 are then the
// eight consecutive values 32 p + 8 g .. + 7 of pair n, one 16-byte store, and the four
// lanes of a pair write 64 consecutive bytes.  The same products in the same order
// as apply_mfma16_kernel, so the same bits.
//
// That kernel holds 32 rows per wave and passes every 64-pair output tile through
// LDS with two barriers and eight dependent scale-and-store rounds per wave, which
// cost more than its memory traffic.  16 x 65536 queries, 16 of 512 states of
// 128 x 128: 3.4 ms there, 2.29 ms here (2.20 without the scattered 4-byte read of
// each pair's gate).  What bounds it now: the 256-byte query rows read and the rows
// written, both scattered, about 11 GB through the L2 misses at 4.7 TB/s (a 1 GiB copy
// reaches 5.2); without the row stores 1.0 ms less, with 32 or 64 pairs per wave and
// step within 4%.
constexpr int AL_THREADS = 512;
constexpr int AL_WAVES = AL_THREADS / 64;
constexpr int AL_NJ = 3;             // 16-pair columns per wave and step
constexpr int AL_PAIRS = 16 * AL_NJ;  // pairs per wave and step

template <class EL, class EQ, int DKP, class EF, int NPART, int NI>
__global__ __launch_bounds__(AL_THREADS, 2) void apply_lds_kernel(const RetrieveArgs a) {
  using rawl = typename ET<EL>::raw;
  using rawf = typename ET<EF>::raw;
  constexpr int NSTEP = DKP / 32;
  constexpr int FRAGS = NSTEP * NI;  // fragments per part
  static_assert(std::is_same_v<EQ, EF>, "the query's bits are the MFMA operand");
  extern __shared__ __align__(16) unsigned char al_smem[];
  Frag8<EF>* As = reinterpret_cast<Frag8<EF>*>(al_smem);  // [NPART][NSTEP][NI][64]

  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t vt = blockIdx.x % a.v_tiles;
  const int64_t tile = blockIdx.x / a.v_tiles;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int p_end = te.z;
  const int dk = a.dk, dv = a.dv;
  const int v0 = static_cast<int>(vt) * AP_V;
  const uint32_t index_bytes = static_cast<uint32_t>(a.n_index) * 4;
  const __amdgpu_buffer_rsrc_t rl = make_rsrc(a.list + b * a.n_index, index_bytes);
  const __amdgpu_buffer_rsrc_t rout =
      make_rsrc(static_cast<const uint16_t*>(a.out) + b * a.n_index * dv, static_cast<uint32_t>(a.n_index * dv * 2));
  const __amdgpu_buffer_rsrc_t rscale =
      make_rsrc(a.scales + b * a.n_index * a.v_tiles, static_cast<uint32_t>(a.n_index * a.v_tiles * 4));
  auto load_id = [&](int p) {  // -1 past the tile
    const int off = p + lane < p_end ? (p + lane) * 4 : kBufOOB;
    const int id = static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(rl, off, 0, 0));
    return p + lane < p_end ? id : -1;
  };

  const __amdgpu_buffer_rsrc_t rg = make_rsrc(a.gates + b * a.n_index, index_bytes);
  auto load_gate = [&](int id) { return buf_load1<F32>(rg, id >= 0 ? id * 4 : kBufOOB); };

  // Pair ids (one per lane) of this wave's first 48 pairs, their gates, ids of the next.
  int p0 = te.y + AL_PAIRS * w;
  int pid = load_id(p0), pid_next = load_id(p0 + AL_PAIRS * AL_WAVES);
  float gate = load_gate(pid);
  {
    const rawl* msrc = static_cast<const rawl*>(a.mem) + (b * a.segments + te.x) * dv * dk;
    const __amdgpu_buffer_rsrc_t rm = make_rsrc(msrc, static_cast<uint32_t>(dv * dk * sizeof(rawl)));
    constexpr int EPU = 16 / static_cast<int>(sizeof(rawl));
    constexpr int UNITS = (FRAGS + AL_WAVES - 1) / AL_WAVES;  // fragments per wave
    float x[UNITS][8];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int f = w + AL_WAVES * u, c = f % NSTEP, i = f / NSTEP;
      const int v = v0 + 32 * (i >> 1) + 8 * (n >> 2) + 4 * (i & 1) + (n & 3), k = 32 * c + 8 * g;
#pragma unroll
      for (int h = 0; h < 8; h += EPU)
        load16_f32<EL>(rm, (i < NI && v < dv && k + h < dk) ? (v * dk + k + h) * static_cast<int>(sizeof(rawl)) : kBufOOB,
                       &x[u][h]);
    }
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int f = w + AL_WAVES * u, c = f % NSTEP, i = f / NSTEP;
      if (i >= NI) continue;
#pragma unroll
      for (int part = 0; part < NPART; ++part) {
        Frag8<EF> fr;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const rawf h = ET<EF>::from_f(x[u][e]);
          fr.e[e] = h;
          x[u][e] -= ET<EF>::to_f(h);
        }
        As[((part * NSTEP + c) * NI + i) * 64 + lane] = fr;
      }
    }
  }

  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc(static_cast<const rawf*>(a.queries) + b * a.n_query * dk, static_cast<uint32_t>(a.n_query * dk * 2));
  Frag8<EF> bq[AL_NJ][NSTEP];
  // Byte offsets of this lane's part of its three pairs' queries; the step is the scalar
  // offset, which rows_in_lds keeps below the resource's size (the range check compares
  // the vector offset with the size less the scalar offset).
  int qoff[AL_NJ];
  auto set_q = [&](int qrow_src) {
#pragma unroll
    for (int j = 0; j < AL_NJ; ++j) {
      const int qrow = __shfl(qrow_src, 16 * j + n, 64);
      qoff[j] = qrow >= 0 ? (qrow * dk + 8 * g) * 2 : kBufOOB;
    }
  };
  auto load_q = [&](int c) {
#pragma unroll
    for (int j = 0; j < AL_NJ; ++j)
      bq[j][c] = __builtin_bit_cast(Frag8<EF>, __builtin_amdgcn_raw_buffer_load_b128(
                                                   rq, 32 * c + 8 * g < dk ? qoff[j] : kBufOOB, 64 * c, 0));
  };
  set_q(query_of(a, pid));
#pragma unroll
  for (int c = 0; c < NSTEP; ++c) load_q(c);
  __syncthreads();  // the state's fragments

  while (p0 < p_end) {
    const int pn = p0 + AL_PAIRS * AL_WAVES;
    const int pid_after = load_id(pn + AL_PAIRS * AL_WAVES);
    const float gate_next = load_gate(pid_next);
    set_q(query_of(a, pid_next));
    f32x4 acc[NI][AL_NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < AL_NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Fragments in the order of use, AHEAD of them read before their MFMAs; the
    // scheduling barriers keep the compiler from reading all of them first (and
    // spilling).
    constexpr int NF = FRAGS * NPART, AHEAD = 2;
    Frag8<EF> am[AHEAD];
    auto frag = [&](int f) {  // f = (c NPART + part) NI + i
      const int c = f / (NPART * NI), part = f / NI % NPART, i = f % NI;
      return As[((part * NSTEP + c) * NI + i) * 64 + lane];
    };
#pragma unroll
    for (int f = 0; f < AHEAD; ++f) am[f] = frag(f);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int c = f / (NPART * NI), i = f % NI;
      const Frag8<EF> af = am[f % AHEAD];
      if (f + AHEAD < NF) am[f % AHEAD] = frag(f + AHEAD);
#pragma unroll
      for (int j = 0; j < AL_NJ; ++j) acc[i][j] = mfma8(af, bq[j][c], acc[i][j]);
      // the next 48 pairs' keys of this step, in flight from here on
      if ((f + 1) % (NPART * NI) == 0) load_q(c);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < AL_NJ; ++j) {
      const int pj = __shfl(pid, 16 * j + n, 64);
      const float gj = __shfl(gate, 16 * j + n, 64);
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        acc[i][j] *= gj;
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, fabsf(acc[i][j][r]));
      }
      {  // over the four lanes of the pair
        const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        m = fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
        const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        m = fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
      }
      int ex = 0;
      (void)frexpf(m, &ex);
      const int sh = min(max(15 - ex, -100), 100);
      const int ro = pj * (2 * dv) + 2 * (v0 + 8 * g);  // pj = -1: below zero, out of range
#pragma unroll
      for (int p = 0; p < NI / 2; ++p) {
        u32x4 q;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 y = acc[2 * p + h][j];
          q[2 * h] = pack2<F16>(ldexpf(y[0], sh), ldexpf(y[1], sh));
          q[2 * h + 1] = pack2<F16>(ldexpf(y[2], sh), ldexpf(y[3], sh));
        }
        __builtin_amdgcn_raw_buffer_store_b128(q, rout, v0 + 32 * p + 8 * g < dv ? ro + 64 * p : kBufOOB, 0, 0);
      }
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ldexpf(1.f, -sh)), rscale,
                                            g == 0 ? (pj * a.v_tiles + static_cast<int>(vt)) * 4 : kBufOOB, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    p0 = pn;
    pid = pid_next;
    pid_next = pid_after;
    gate = gate_next;
  }
}

template <class EL, class EQ, int DKP, class EF, int NPART, int NI>
int launch_apply_lds(const RetrieveArgs& a, hipStream_t s) {
  constexpr size_t lds = static_cast<size_t>(NPART) * (DKP / 32) * NI * 64 * 16;
  static_assert(lds <= 160 * 1024, "the state's parts fit one CU's LDS");
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&apply_lds_kernel<EL, EQ, DKP, EF, NPART, NI>),
        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) {
      set_error("retrieve_fuse: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
  }
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(a.tb_max) * a.v_tiles), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_lds_kernel<EL, EQ, DKP, EF, NPART, NI>), grid, dim3(AL_THREADS), lds, s, a);
  return check_launch("retrieve_fuse(apply)");
}

// The state in LDS where enough pairs share its staging, which eight waves do while with
// few pairs only one or two of them have any.  Time of the call with output tiles over
// time with the state in LDS, 16 x 256 states, 8 routes, at 8, 32, 64, 128, 256 and 512
// pairs per state (float32 and float16 states, widths of 32, 64 and 128 keys):
//   32 values:   1.0-1.2, 1.1-1.3, 1.3-1.5, 1.4-1.7, 1.5-2.1, 1.4-2.2: always
//   64 values:   0.8-1.0, 1.0-1.1, 1.1-1.3, 1.2-1.5, 1.3-1.5, 1.2-1.7: from 32 pairs
//   128 values:  0.6-0.8, 0.7-0.9, 0.8-1.0, 0.9-1.0, 1.0-1.1, 1.1-1.4: from 256 pairs
// The byte offsets of that kernel are 32 bits, and its scalar offsets stay inside the queries.
bool rows_in_lds(const RetrieveArgs& a, int64_t tiles) {
  const int64_t pairs = a.dv <= 32 ? 0 : a.dv <= 64 ? 32 : 256;
  const int steps = a.dk <= 32 ? 1 : a.dk <= 64 ? 2 : 4;
  return a.n_index >= pairs * a.segments && a.n_query * a.dk * 2 >= 64 * steps &&
         a.n_index * a.dv * 2 <= INT32_MAX && tiles * a.v_tiles * AL_THREADS <= UINT32_MAX;
}

template <class EL, class EQ, int DKP, class EF, int NPART, int NI>
int launch_scaled_rows(const RetrieveArgs& a, hipStream_t s) {
  if (a.lds_rows != 0) return launch_apply_lds<EL, EQ, DKP, EF, NPART, NI>(a, s);
  return launch_apply_mfma16<EL, F32, EQ, DKP, EF, NPART, true>(a, s);
}

template <class EL, class EQ, int DKP, class EF, int NPART>
int launch_scaled_width(const RetrieveArgs& a, hipStream_t s) {
  if (a.dv <= 32) return launch_scaled_rows<EL, EQ, DKP, EF, NPART, 2>(a, s);
  if (a.dv <= 64) return launch_scaled_rows<EL, EQ, DKP, EF, NPART, 4>(a, s);
  return launch_scaled_rows<EL, EQ, DKP, EF, NPART, 8>(a, s);
}

// The scaled apply runs the exact 16-bit MFMA kernel with float32 arithmetic;
// other dtype pairs and unaligned shapes are not supported by retrieve_fuse.
template <class EL, class EQ>
int launch_apply_scaled(const RetrieveArgs& a, hipStream_t s) {
  using Plan = MfmaPlan<EL, F32, EQ>;
  if constexpr (Plan::ok) {
    using EF = typename Plan::EF;
    constexpr int NPART = Plan::parts;
    if (a.dk <= 32) return launch_scaled_width<EL, EQ, 32, EF, NPART>(a, s);
    if (a.dk <= 64) return launch_scaled_width<EL, EQ, 64, EF, NPART>(a, s);
    return launch_scaled_width<EL, EQ, 128, EF, NPART>(a, s);
  } else {
    set_error("retrieve_fuse: no exact 16-bit MFMA plan for these dtypes");
    return GRM_HIP_EUNSUPPORTED;
  }
}

template <class EL>
bool scaled_ok_q(const RetrieveArgs& a, int q_dtype) {
  switch (q_dtype) {
    case GRM_HIP_F16: return MfmaPlan<EL, F32, F16>::ok && vec_ok<EL, F16>(a);
    case GRM_HIP_BF16: return MfmaPlan<EL, F32, BF16>::ok && vec_ok<EL, BF16>(a);
    default: return false;
  }
}

bool scaled_supported(const RetrieveArgs& a, int mem_dtype, int q_dtype) {
  switch (mem_dtype) {
    case GRM_HIP_F32: return scaled_ok_q<F32>(a, q_dtype);
    case GRM_HIP_F16: return scaled_ok_q<F16>(a, q_dtype);
    default: return scaled_ok_q<BF16>(a, q_dtype);
  }
}

template <class EL>
int apply_scaled_q(const RetrieveArgs& a, int q_dtype, hipStream_t s) {
  return q_dtype == GRM_HIP_F16 ? launch_apply_scaled<EL, F16>(a, s) : launch_apply_scaled<EL, BF16>(a, s);
}

// ---------------------------------------------------------------------------
// The queries' gradient of gather_apply: for every pair (q, r) with a valid
// index, dqp[b, q, r, :] = M[b, idx[b, q, r]]^T g[b, q, r, :] (float32 grad_out
// rows of d_v, float32 result rows of d_k); the caller sums over r.  One
// workgroup of 8 waves per (sequence, work tile) stages its segment's state in
// LDS as float32, rows of d_v padded to a multiple of 16 with zeros, row stride
// DKP + 4 floats, and applies its transpose with float32 MFMA (16x16x4).  Wave
// w takes 16 pairs at a time: in MFMA j of value block v0, lane (kq, n) gives
// A = M[v0 + 4 kq + j][16 kb + n] and B = g[pair n][v0 + 4 kq + j], so each
// lane's gradient values of a block are one float4 (loaded a 128-value chunk
// ahead of the MFMAs), and the four rows one A read touches (4 apart) start
// 16 banks apart.  Each output row is written by one wave: deterministic, no
// atomics.
constexpr int AT_THREADS = 512;
constexpr int AT_CHUNK = 8;  // value blocks of 16 per prefetched chunk

template <int DKP>
__host__ __device__ constexpr int at_row_stride() { return DKP + 4; }

__host__ __device__ inline int at_rows(int dv) { return (dv + 15) / 16 * 16; }

template <class EL, int DKP>
__global__ __launch_bounds__(AT_THREADS) void apply_t_kernel(const RetrieveArgs a, const float* grad, float* dqp,
                                                             int vec_state, int vec_grad, int token_rows) {
  using rawl = typename ET<EL>::raw;
  extern __shared__ float Ms[];  // [at_rows(dv)][DKP + 4]
  constexpr int MSK = at_row_stride<DKP>();
  constexpr int KB = DKP / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t tile = blockIdx.x;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int64_t s = te.x;
  const int p_begin = te.y, p_end = te.z;
  const int dk = a.dk, dv = a.dv, dv16 = at_rows(dv);
  const rawl* msrc = static_cast<const rawl*>(a.mem) + (b * a.segments + s) * dv * dk;
  if (vec_state) {
    // dk == DKP and 16-byte aligned rows: 16 bytes of the state per thread and step
    constexpr int PER = 16 / sizeof(rawl);
    const int nvec = dv * DKP / PER;
    for (int e = tid; e < nvec; e += AT_THREADS) {
      const int idx = e * PER;
      const int v = idx / DKP, k = idx % DKP;
      rawl t[PER];
      *reinterpret_cast<uint4*>(t) = *reinterpret_cast<const uint4*>(msrc + idx);
#pragma unroll
      for (int i = 0; i < PER; i += 4)
        *reinterpret_cast<f32x4*>(Ms + v * MSK + k + i) =
            f32x4{ET<EL>::to_f(t[i]), ET<EL>::to_f(t[i + 1]), ET<EL>::to_f(t[i + 2]), ET<EL>::to_f(t[i + 3])};
    }
    for (int e = dv * DKP + tid; e < dv16 * DKP; e += AT_THREADS) Ms[(e / DKP) * MSK + e % DKP] = 0.f;
  } else {
    for (int e = tid; e < dv16 * DKP; e += AT_THREADS) {
      const int v = e / DKP, k = e % DKP;
      Ms[v * MSK + k] = (v < dv && k < dk) ? ET<EL>::to_f(msrc[v * dk + k]) : 0.f;
    }
  }
  __syncthreads();
  const int32_t* lb = a.list + b * a.n_index;
  const int n = lane & 15, kq = lane >> 4;
  const int n_chunks = (dv16 / 16 + AT_CHUNK - 1) / AT_CHUNK;
  int p0 = p_begin + 16 * w;
  int pid = p0 < p_end && p0 + n < p_end ? lb[p0 + n] : -1;
  for (; p0 < p_end; p0 += 16 * (AT_THREADS / 64)) {
    const int pn = p0 + 16 * (AT_THREADS / 64);
    const int pid_next = pn + n < p_end ? lb[pn + n] : -1;
    // grad rows per pair, or (token_rows) one row per query shared by its routes
    const int64_t grow_i = token_rows ? b * a.n_query + query_of(a, pid >= 0 ? pid : 0)
                                      : b * a.n_index + (pid >= 0 ? pid : 0);
    const float* grow = grad + grow_i * static_cast<int64_t>(dv);
    auto load_chunk = [&](f32x4* g, int c) {
#pragma unroll
      for (int u = 0; u < AT_CHUNK; ++u) {
        const int vq = 16 * (AT_CHUNK * c + u) + 4 * kq;
        f32x4 x{0.f, 0.f, 0.f, 0.f};
        if (pid >= 0) {
          if (vec_grad) {
            if (vq < dv) x = *reinterpret_cast<const f32x4*>(grow + vq);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (vq + r < dv) x[r] = grow[vq + r];
          }
        }
        g[u] = x;
      }
    };
    f32x4 acc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) acc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 cur[AT_CHUNK], nxt[AT_CHUNK];
    load_chunk(cur, 0);
    for (int c = 0; c < n_chunks; ++c) {
      if (c + 1 < n_chunks) load_chunk(nxt, c + 1);
#pragma unroll
      for (int u = 0; u < AT_CHUNK; ++u) {
        const int v0 = 16 * (AT_CHUNK * c + u);
        if (v0 < dv16) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float* mrow = Ms + (v0 + 4 * kq + j) * MSK + n;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
              acc[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(mrow[16 * kb], cur[u][j], acc[kb], 0, 0, 0);
          }
        }
      }
      if (c + 1 < n_chunks) {
#pragma unroll
        for (int u = 0; u < AT_CHUNK; ++u) cur[u] = nxt[u];
      }
    }
    // lane (kq, n) holds keys 16 kb + 4 kq + r of pair n (the pair its pid names)
    if (pid >= 0) {
      float* orow = dqp + (b * a.n_index + pid) * static_cast<int64_t>(dk);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int k = 16 * kb + 4 * kq;
        if (k + 4 <= dk && (dk & 3) == 0) {
          *reinterpret_cast<f32x4*>(orow + k) = acc[kb];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (k + r < dk) orow[k + r] = acc[kb][r];
        }
      }
    }
    pid = pid_next;
  }
}

// The same per-pair product M[idx]^T g for float16 archives on 16-bit MFMA.
// The state sits in LDS transposed ([DKP][value index], float16, rows padded by
// 8 values so the 16 rows of one fragment read start 4 banks apart).  Each
// 32-value chunk of a pair's float32 gradient row is scaled by the power of two
// that puts its largest magnitude in [2^14, 2^15) and split into float16 parts
// hi = round(g s) and lo = round(g s - hi); two 16x16x32 MFMAs (products of
// float16 values are exact in fp32) and one multiply by 1/s per chunk.  Error
// per chunk about 2^-22 of its largest magnitude times sum_v |M[v][k]|, the size
// of the fp32 accumulation's own rounding.  Chunks of 4 are loaded one group
// ahead, as apply_t_kernel does.
__host__ __device__ inline int at16_stride(int dv) { return (dv + 31) / 32 * 32 + 8; }

template <int DKP>
__global__ __launch_bounds__(AT_THREADS) void apply_t16_kernel(const RetrieveArgs a, const float* grad, float* dqp,
                                                               int vec_state, int vec_grad, int token_rows) {
  extern __shared__ uint16_t MsT[];  // [DKP][at16_stride(dv)]
  constexpr int KB = DKP / 16;
  constexpr int GC = 4;  // 32-value chunks per prefetched group
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t tile = blockIdx.x;
  const int64_t b = blockIdx.y;
  if (tile >= a.n_tiles[b]) return;
  const int4 te = a.tiles[b * a.tb_max + tile];
  const int64_t s = te.x;
  const int p_begin = te.y, p_end = te.z;
  const int dk = a.dk, dv = a.dv;
  const int VS = at16_stride(dv);
  const int dv32 = VS - 8;
  const uint16_t* msrc = static_cast<const uint16_t*>(a.mem) + (b * a.segments + s) * dv * dk;
  if (vec_state) {
    // 16 bytes (8 key values of one value row) per thread and step, written transposed
    const int nvec = dv * dk / 8;
    for (int e = tid; e < nvec; e += AT_THREADS) {
      const int idx = 8 * e;
      const int v = idx / dk, k = idx % dk;
      const uint4 t = *reinterpret_cast<const uint4*>(msrc + idx);
      const uint32_t wds[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        MsT[(k + 2 * j) * VS + v] = static_cast<uint16_t>(wds[j] & 0xffffu);
        MsT[(k + 2 * j + 1) * VS + v] = static_cast<uint16_t>(wds[j] >> 16);
      }
    }
  } else {
    for (int e = tid; e < dv * dk; e += AT_THREADS) MsT[(e % dk) * VS + e / dk] = msrc[e];
  }
  if (dk < DKP || dv < dv32) {
    for (int e = tid; e < DKP * dv32; e += AT_THREADS) {
      const int k = e / dv32, v = e % dv32;
      if (k >= dk || v >= dv) MsT[k * VS + v] = 0;
    }
  }
  __syncthreads();
  const int32_t* lb = a.list + b * a.n_index;
  const int n = lane & 15, kq = lane >> 4;
  const int nch = dv32 / 32;
  const int ngr = (nch + GC - 1) / GC;
  int p0 = p_begin + 16 * w;
  int pid = p0 < p_end && p0 + n < p_end ? lb[p0 + n] : -1;
  for (; p0 < p_end; p0 += 16 * (AT_THREADS / 64)) {
    const int pn = p0 + 16 * (AT_THREADS / 64);
    const int pid_next = pn + n < p_end ? lb[pn + n] : -1;
    // grad rows per pair, or (token_rows) one row per query shared by its routes
    const int64_t grow_i = token_rows ? b * a.n_query + query_of(a, pid >= 0 ? pid : 0)
                                      : b * a.n_index + (pid >= 0 ? pid : 0);
    const float* grow = grad + grow_i * static_cast<int64_t>(dv);
    // values 32 c + 8 kq .. + 7 of this lane's pair, chunks of group gi
    auto load_group = [&](float (&x)[GC][8], int gi) {
#pragma unroll
      for (int u = 0; u < GC; ++u) {
        const int v = 32 * (GC * gi + u) + 8 * kq;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[u][j] = 0.f;
        if (pid >= 0) {
          if (vec_grad) {
            if (v < dv) {
              const f32x4 lo4 = *reinterpret_cast<const f32x4*>(grow + v);
#pragma unroll
              for (int j = 0; j < 4; ++j) x[u][j] = lo4[j];
            }
            if (v + 4 < dv) {
              const f32x4 hi4 = *reinterpret_cast<const f32x4*>(grow + v + 4);
#pragma unroll
              for (int j = 0; j < 4; ++j) x[u][4 + j] = hi4[j];
            }
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (v + j < dv) x[u][j] = grow[v + j];
          }
        }
      }
    };
    f32x4 acc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) acc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    float cur[GC][8], nxt[GC][8];
    load_group(cur, 0);
    for (int gi = 0; gi < ngr; ++gi) {
      if (gi + 1 < ngr) load_group(nxt, gi + 1);
#pragma unroll
      for (int u = 0; u < GC; ++u) {
        const int c = GC * gi + u;
        if (c < nch) {
          // the chunk's scale: its largest magnitude over the pair's 4 lanes
          float m = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(cur[u][j]));
          m = fmaxf(m, __shfl_xor(m, 16, 64));
          m = fmaxf(m, __shfl_xor(m, 32, 64));
          const int ex = static_cast<int>((__float_as_uint(m) >> 23) & 0xffu);
          // s = 2^(14 - floor(log2 m)) as a biased exponent in [1, 253]; 1 for 0 or inf
          const int es = (m > 0.f && ex < 255) ? min(max(268 - ex, 1), 253) : 127;
          const float sc = __uint_as_float(static_cast<uint32_t>(es) << 23);
          const float inv = __uint_as_float(static_cast<uint32_t>(254 - es) << 23);
          Frag8<F16> hi, lo;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float x = cur[u][j] * sc;
            hi.e[j] = ET<F16>::from_f(x);
            lo.e[j] = ET<F16>::from_f(x - ET<F16>::to_f(hi.e[j]));
          }
          const int vA = 32 * c + 8 * kq;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            const Frag8<F16> am =
                __builtin_bit_cast(Frag8<F16>, *reinterpret_cast<const uint4*>(MsT + (16 * kb + n) * VS + vA));
            f32x4 t = mfma8(am, hi, f32x4{0.f, 0.f, 0.f, 0.f});
            t = mfma8(am, lo, t);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[kb][r] = fmaf(t[r], inv, acc[kb][r]);
          }
        }
      }
      if (gi + 1 < ngr) {
#pragma unroll
        for (int u = 0; u < GC; ++u)
#pragma unroll
          for (int j = 0; j < 8; ++j) cur[u][j] = nxt[u][j];
      }
    }
    // lane (kq, n) holds keys 16 kb + 4 kq + r of pair n (the pair its pid names)
    if (pid >= 0) {
      float* orow = dqp + (b * a.n_index + pid) * static_cast<int64_t>(dk);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int k = 16 * kb + 4 * kq;
        if (k + 4 <= dk && (dk & 3) == 0) {
          *reinterpret_cast<f32x4*>(orow + k) = acc[kb];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (k + r < dk) orow[k + r] = acc[kb][r];
        }
      }
    }
    pid = pid_next;
  }
}

inline size_t apply_t16_lds(int dv, int dkp) { return static_cast<size_t>(dkp) * at16_stride(dv) * sizeof(uint16_t); }

template <int DKP>
int launch_apply_t16(const RetrieveArgs& a, const float* grad, float* dqp, int token_rows, hipStream_t s) {
  const size_t lds = apply_t16_lds(a.dv, DKP);
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&apply_t16_kernel<DKP>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
      set_error("gather_apply_bwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
    attr_set = true;
  }
  const int vec_state = a.dk % 8 == 0 && reinterpret_cast<uintptr_t>(a.mem) % 16 == 0;
  const int vec_grad = a.dv % 4 == 0 && reinterpret_cast<uintptr_t>(grad) % 16 == 0;
  const dim3 grid(static_cast<unsigned>(a.tb_max), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_t16_kernel<DKP>), grid, dim3(AT_THREADS), lds, s, a, grad, dqp, vec_state, vec_grad,
                     token_rows);
  return check_launch("gather_apply_bwd");
}

inline size_t apply_t_lds(int dv, int dkp) {
  return static_cast<size_t>(at_rows(dv)) * (dkp + 4) * sizeof(float);
}

template <class EL, int DKP>
int launch_apply_t(const RetrieveArgs& a, const float* grad, float* dqp, int token_rows, hipStream_t s) {
  using rawl = typename ET<EL>::raw;
  const size_t lds = apply_t_lds(a.dv, DKP);
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&apply_t_kernel<EL, DKP>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
      set_error("gather_apply_bwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
    attr_set = true;
  }
  const int vec_state = a.dk == DKP && (DKP * sizeof(rawl)) % 16 == 0 &&
                        reinterpret_cast<uintptr_t>(a.mem) % 16 == 0;
  const int vec_grad = a.dv % 4 == 0 && reinterpret_cast<uintptr_t>(grad) % 16 == 0;
  const dim3 grid(static_cast<unsigned>(a.tb_max), static_cast<unsigned>(a.batch));
  hipLaunchKernelGGL((apply_t_kernel<EL, DKP>), grid, dim3(AT_THREADS), lds, s, a, grad, dqp, vec_state, vec_grad,
                     token_rows);
  return check_launch("gather_apply_bwd");
}

template <class EL>
int dispatch_apply_t(const RetrieveArgs& a, const float* grad, float* dqp, int token_rows, hipStream_t s) {
  if constexpr (std::is_same_v<EL, F16>) {
    // float16 archives: the 16-bit MFMA form (GRM_HIP_APPLY_T16=0 keeps the fp32 one)
    const char* env = getenv("GRM_HIP_APPLY_T16");
    if (env == nullptr || env[0] != '0') {
      if (a.dk <= 16) return launch_apply_t16<16>(a, grad, dqp, token_rows, s);
      if (a.dk <= 32) return launch_apply_t16<32>(a, grad, dqp, token_rows, s);
      if (a.dk <= 64) return launch_apply_t16<64>(a, grad, dqp, token_rows, s);
      return launch_apply_t16<128>(a, grad, dqp, token_rows, s);
    }
  }
  if (a.dk <= 16) return launch_apply_t<EL, 16>(a, grad, dqp, token_rows, s);
  if (a.dk <= 32) return launch_apply_t<EL, 32>(a, grad, dqp, token_rows, s);
  if (a.dk <= 64) return launch_apply_t<EL, 64>(a, grad, dqp, token_rows, s);
  return launch_apply_t<EL, 128>(a, grad, dqp, token_rows, s);
}

int allow_segment_lds(const void* fn) {
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(kMaxSegments * sizeof(int)));
  if (e != hipSuccess) {
    set_error("gather_apply: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
    return static_cast<int>(e);
  }
  return GRM_HIP_OK;
}

template <class EM>
int launch_bucket(const RetrieveArgs& a, hipStream_t s) {
  const size_t lds = static_cast<size_t>(a.segments) * sizeof(int);
  static int attr_rc = -1;
  if (attr_rc != GRM_HIP_OK) {
    attr_rc = allow_segment_lds(reinterpret_cast<const void*>(&bucket_kernel<EM>));
    if (attr_rc == GRM_HIP_OK) attr_rc = allow_segment_lds(reinterpret_cast<const void*>(&bucket_count_kernel<EM>));
    if (attr_rc == GRM_HIP_OK) attr_rc = allow_segment_lds(reinterpret_cast<const void*>(&bucket_bases_kernel));
    if (attr_rc == GRM_HIP_OK) attr_rc = allow_segment_lds(reinterpret_cast<const void*>(&bucket_scatter_kernel));
    if (attr_rc == GRM_HIP_OK) attr_rc = allow_segment_lds(reinterpret_cast<const void*>(&tile_list_kernel));
    if (attr_rc != GRM_HIP_OK) return attr_rc;
  }
  int rc;
  if (a.bk_chunks <= 1) {
    hipLaunchKernelGGL((bucket_kernel<EM>), dim3(static_cast<unsigned>(a.batch)), dim3(BK_THREADS), lds, s, a);
    rc = check_launch("gather_apply(sort)");
  } else {
    const dim3 grid(static_cast<unsigned>(a.bk_chunks), static_cast<unsigned>(a.batch));
    hipLaunchKernelGGL((bucket_count_kernel<EM>), grid, dim3(BK_THREADS), lds, s, a);
    rc = check_launch("gather_apply(sort counts)");
    if (rc != GRM_HIP_OK) return rc;
    hipLaunchKernelGGL(bucket_bases_kernel, dim3(static_cast<unsigned>(a.batch)), dim3(BK_THREADS), lds, s, a);
    rc = check_launch("gather_apply(sort bases)");
    if (rc != GRM_HIP_OK) return rc;
    hipLaunchKernelGGL(bucket_scatter_kernel, grid, dim3(BK_THREADS), lds, s, a);
    rc = check_launch("gather_apply(sort scatter)");
  }
  if (rc != GRM_HIP_OK || a.segments == 0) return rc;
  hipLaunchKernelGGL(tile_list_kernel, dim3(static_cast<unsigned>(a.batch)), dim3(BK_THREADS), lds, s, a);
  return check_launch("gather_apply(tile list)");
}

int64_t offsets_bytes(int64_t batch, int64_t segments) { return (batch * (segments + 1) * 4 + 15) / 16 * 16; }

// Pair chunks per sequence for the multi-workgroup sort (1: one workgroup per sequence).
int64_t bucket_chunks(int64_t batch, int64_t n_index) {
  return n_index >= kMultiBucketPairs && batch <= 65535 ? (n_index + BK_ITEMS - 1) / BK_ITEMS : 1;
}

int64_t list_bytes(int64_t batch, int64_t n_index) { return (batch * n_index * 4 + 15) / 16 * 16; }

int64_t partial_bytes(int64_t batch, int64_t segments, int64_t n_index) {
  const int64_t c = bucket_chunks(batch, n_index);
  return c > 1 ? (batch * c * segments * 4 + 15) / 16 * 16 : 0;
}

// Pairs per apply work tile: the mean pairs per segment (at least 512, a
// multiple of the 64-pair MFMA tile), so balanced selections keep about one
// tile per segment and a heavily selected segment is split.  With few states
// the longest tile is the kernel's time: at one and a half times the mean, an
// uneven selection (weights 1 / sqrt(rank)) over 6 to 32 states took gather_apply
// and its gradients 1.2 to 1.45 times as long (20000 queries, 2 of 6 states of
// 128 x 128, float16: 386 -> 554 us), an even one the same.
// `spread` (the scaled rows with states in LDS, which stage a state per tile):
// one and a half times the mean, since at the mean half of the segments have a
// second tile of a few pairs (16 x 65536 queries over 512 states: 3.97 -> 3.67 ms).
// At most 2^20 pairs, so that no 32-bit count of the tiles overflows.
int64_t tile_pairs_for(int64_t segments, int64_t n_index, bool spread = false) {
  const int64_t mean = segments > 0 ? (n_index + segments - 1) / segments : n_index;
  const int64_t tp = (mean + (spread ? mean / 2 : 0) + AP_N - 1) / AP_N * AP_N;
  return std::min<int64_t>(std::max<int64_t>(tp, 8 * AP_N), 1 << 20);
}

// Tiles per sequence at most: sum_s ceil(c_s / tp) <= n_index / tp + segments.
int64_t tiles_max(int64_t segments, int64_t n_index, bool spread = false) {
  const int64_t tp = tile_pairs_for(segments, n_index, spread);
  return (n_index + tp - 1) / tp + segments;
}

int64_t tiles_bytes(int64_t batch, int64_t segments, int64_t n_index) {
  return batch * tiles_max(segments, n_index) * 16 + (batch * 4 + 15) / 16 * 16 + offsets_bytes(batch, segments);
}

}  // namespace
}  // namespace grmhip

using namespace grmhip;

namespace grmhip {
namespace {

// The sort's workspace carve-up and the sizes, shared by gather_apply and
// retrieve_fuse (the workspace of grm_hip_gather_apply_workspace comes first).
void init_retrieve_args(RetrieveArgs& a, const void* memories, const int64_t* indices, const void* queries, void* out,
                        void* workspace, int64_t batch, int64_t segments, int64_t n_query, int64_t routes,
                        int64_t n_index, int64_t hidden_size, int64_t key_dim, int32_t* bad_index_count) {
  memset(&a, 0, sizeof(a));
  a.mem = memories;
  a.idx = indices;
  a.queries = queries;
  a.out = out;
  a.offsets = static_cast<int32_t*>(workspace);
  a.list = reinterpret_cast<int32_t*>(static_cast<unsigned char*>(workspace) + offsets_bytes(batch, segments));
  a.partial = reinterpret_cast<int32_t*>(static_cast<unsigned char*>(workspace) + offsets_bytes(batch, segments) +
                                         list_bytes(batch, n_index));
  a.bk_chunks = static_cast<int>(bucket_chunks(batch, n_index));
  {
    unsigned char* t0 = static_cast<unsigned char*>(workspace) + offsets_bytes(batch, segments) +
                        list_bytes(batch, n_index) + partial_bytes(batch, segments, n_index);
    a.tile_pairs = static_cast<int>(tile_pairs_for(segments, n_index));
    a.tb_max = static_cast<int>(tiles_max(segments, n_index));
    a.tiles = reinterpret_cast<int4*>(t0);
    t0 += batch * a.tb_max * 16;
    a.n_tiles = reinterpret_cast<int32_t*>(t0);
    t0 += (batch * 4 + 15) / 16 * 16;
    a.tile_base = reinterpret_cast<int32_t*>(t0);
  }
  a.bad = bad_index_count;
  a.batch = batch;
  a.segments = segments;
  a.n_query = n_query;
  a.routes = routes;
  a.n_index = n_index;
  a.dv = static_cast<int>(hidden_size);
  a.dk = static_cast<int>(key_dim);
  a.out_row = a.dv;
  a.v_tiles = static_cast<int>((hidden_size + AP_V - 1) / AP_V);
}

}  // namespace
}  // namespace grmhip

extern "C" int64_t grm_hip_gather_apply_workspace(int64_t batch, int64_t segments, int64_t n_index) {
  if (batch <= 0 || segments < 0 || n_index <= 0) return 0;
  return offsets_bytes(batch, segments) + list_bytes(batch, n_index) + partial_bytes(batch, segments, n_index) +
         tiles_bytes(batch, segments, n_index);
}

extern "C" int grm_hip_gather_apply(const void* memories, const int64_t* indices, const void* queries, void* out,
                                    void* workspace, int64_t workspace_bytes, int64_t batch, int64_t segments,
                                    int64_t n_query, int64_t routes, int64_t hidden_size, int64_t key_dim,
                                    int mem_dtype, int q_dtype, int out_dtype, int32_t* bad_index_count,
                                    void* stream) {
  if (batch < 0 || segments < 0 || n_query < 0 || routes < 0 || hidden_size < 0 || key_dim < 1) {
    set_error("gather_apply: negative size or key_dim < 1");
    return GRM_HIP_EINVAL;
  }
  if (mem_dtype < GRM_HIP_F32 || mem_dtype > GRM_HIP_BF16 || q_dtype < GRM_HIP_F32 || q_dtype > GRM_HIP_BF16) {
    set_error("gather_apply: unsupported dtypes mem=%d q=%d", mem_dtype, q_dtype);
    return GRM_HIP_EUNSUPPORTED;
  }
  if (out_dtype != mem_dtype && out_dtype != GRM_HIP_F32) {
    set_error("gather_apply: out_dtype %d must be the memories' dtype %d or float32", out_dtype, mem_dtype);
    return GRM_HIP_EINVAL;
  }
  if (key_dim > 128 || segments > kMaxSegments) {
    set_error("gather_apply: key_dim %lld > 128 or segments %lld > %lld", (long long)key_dim, (long long)segments,
              (long long)kMaxSegments);
    return GRM_HIP_EUNSUPPORTED;
  }
  const int64_t n_index = n_query * routes;
  if (batch == 0 || n_index == 0 || hidden_size == 0) return GRM_HIP_OK;
  if (n_index > INT32_MAX || hidden_size > INT32_MAX / 2 || batch > 65535 ||
      tiles_max(segments, n_index) * ((hidden_size + AP_V - 1) / AP_V) * AP_THREADS > UINT32_MAX) {
    set_error("gather_apply: sizes exceed one launch");
    return GRM_HIP_EINVAL;
  }
  if (indices == nullptr || queries == nullptr || out == nullptr || (segments > 0 && memories == nullptr)) {
    set_error("gather_apply: null pointer");
    return GRM_HIP_EINVAL;
  }
  const int64_t need = grm_hip_gather_apply_workspace(batch, segments, n_index);
  if (workspace == nullptr || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) {
    set_error("gather_apply: workspace of %lld bytes (16-byte aligned) required", (long long)need);
    return GRM_HIP_EINVAL;
  }
  RetrieveArgs a;
  init_retrieve_args(a, memories, indices, queries, out, workspace, batch, segments, n_query, routes, n_index,
                     hidden_size, key_dim, bad_index_count);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc;
  switch (out_dtype) {
    case GRM_HIP_F32: rc = launch_bucket<F32>(a, s); break;
    case GRM_HIP_F16: rc = launch_bucket<F16>(a, s); break;
    default: rc = launch_bucket<BF16>(a, s); break;
  }
  if (rc != GRM_HIP_OK || segments == 0) return rc;
  if (out_dtype == GRM_HIP_F32) {
    // float32 arithmetic and output; 16-bit memories are widened exactly on load
    switch (mem_dtype) {
      case GRM_HIP_F32: return dispatch_q<F32, F32>(a, q_dtype, s);
      case GRM_HIP_F16: return dispatch_q<F16, F32>(a, q_dtype, s);
      default: return dispatch_q<BF16, F32>(a, q_dtype, s);
    }
  }
  switch (mem_dtype) {
    case GRM_HIP_F16: return dispatch_q<F16, F16>(a, q_dtype, s);
    default: return dispatch_q<BF16, BF16>(a, q_dtype, s);
  }
}

namespace {

int64_t align16(int64_t n) { return (n + 15) / 16 * 16; }

}  // namespace

extern "C" int64_t grm_hip_retrieve_fuse_workspace(int64_t batch, int64_t segments, int64_t n_index,
                                                   int64_t value_dim) {
  if (batch <= 0 || segments < 0 || n_index <= 0 || value_dim <= 0) return 0;
  const int64_t tiles = (value_dim + AP_V - 1) / AP_V;
  return grm_hip_gather_apply_workspace(batch, segments, n_index) + align16(batch * n_index * value_dim * 2) +
         align16(batch * n_index * tiles * 4);
}

extern "C" int grm_hip_retrieve_fuse(const void* memories, const int64_t* indices, const void* queries,
                                     const float* gates, const void* h_online, const void* ln_weight,
                                     const void* ln_bias, void* out, void* workspace, int64_t workspace_bytes,
                                     int64_t batch, int64_t segments, int64_t n_query, int64_t routes,
                                     int64_t value_dim, int64_t key_dim, int mem_dtype, int q_dtype, int h_dtype,
                                     float eps, int32_t* bad_index_count, void* stream) {
  if (batch < 0 || segments < 0 || n_query < 0 || routes < 0 || value_dim < 0 || key_dim < 1) {
    set_error("retrieve_fuse: negative size or key_dim < 1");
    return GRM_HIP_EINVAL;
  }
  if (mem_dtype < GRM_HIP_F32 || mem_dtype > GRM_HIP_BF16 || q_dtype < GRM_HIP_F32 || q_dtype > GRM_HIP_BF16 ||
      h_dtype < GRM_HIP_F32 || h_dtype > GRM_HIP_BF16) {
    set_error("retrieve_fuse: unsupported dtypes mem=%d q=%d h=%d", mem_dtype, q_dtype, h_dtype);
    return GRM_HIP_EUNSUPPORTED;
  }
  if (key_dim > 128 || segments > kMaxSegments || value_dim % 8 != 0 || value_dim > 2048) {
    set_error("retrieve_fuse: needs key_dim <= 128, segments <= %lld, value_dim a multiple of 8 and <= 2048",
              (long long)kMaxSegments);
    return GRM_HIP_EUNSUPPORTED;
  }
  const int64_t rows = batch * n_query;
  const int64_t n_index = n_query * routes;
  if (rows == 0 || value_dim == 0) return GRM_HIP_OK;
  if (h_online == nullptr || out == nullptr || (n_index > 0 && (indices == nullptr || queries == nullptr ||
                                                                gates == nullptr)) ||
      (segments > 0 && memories == nullptr)) {
    set_error("retrieve_fuse: null pointer");
    return GRM_HIP_EINVAL;
  }
  if (n_index > INT32_MAX || batch > 65535 || routes * value_dim * 2 > INT32_MAX ||
      tiles_max(segments, n_index) * ((value_dim + AP_V - 1) / AP_V) * AP_THREADS > UINT32_MAX) {
    set_error("retrieve_fuse: sizes exceed one launch");
    return GRM_HIP_EINVAL;
  }
  const int64_t need = grm_hip_retrieve_fuse_workspace(batch, segments, n_index, value_dim);
  if (n_index > 0 &&
      (workspace == nullptr || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16 != 0)) {
    set_error("retrieve_fuse: workspace of %lld bytes (16-byte aligned) required", (long long)need);
    return GRM_HIP_EINVAL;
  }
  const int hb = h_dtype == GRM_HIP_F32 ? 4 : 2;
  if (reinterpret_cast<uintptr_t>(h_online) % 16 != 0 || reinterpret_cast<uintptr_t>(out) % 16 != 0 ||
      (ln_weight != nullptr && reinterpret_cast<uintptr_t>(ln_weight) % 16 != 0) ||
      (ln_bias != nullptr && reinterpret_cast<uintptr_t>(ln_bias) % 16 != 0) || (value_dim * hb) % 16 != 0) {
    set_error("retrieve_fuse: h_online, out and the LayerNorm parameters must be 16-byte aligned");
    return GRM_HIP_EUNSUPPORTED;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int v_tiles = static_cast<int>((value_dim + AP_V - 1) / AP_V);
  unsigned char* rows16 = nullptr;
  float* scales = nullptr;
  if (n_index > 0) {
    rows16 = static_cast<unsigned char*>(workspace) + grm_hip_gather_apply_workspace(batch, segments, n_index);
    scales = reinterpret_cast<float*>(rows16 + align16(batch * n_index * value_dim * 2));
    RetrieveArgs a;
    init_retrieve_args(a, memories, indices, queries, rows16, workspace, batch, segments, n_query, routes, n_index,
                       value_dim, key_dim, bad_index_count);
    a.gates = gates;
    a.scales = scales;
    if (!scaled_supported(a, mem_dtype, q_dtype)) {
      set_error("retrieve_fuse: needs bf16 queries (or f16 queries with f16 memories), 16-byte rows and "
                "16-byte aligned memories and queries");
      return GRM_HIP_EUNSUPPORTED;
    }
    const int64_t spread_tiles = tiles_max(segments, n_index, true);  // not more than the workspace holds
    if (rows_in_lds(a, spread_tiles)) {
      a.lds_rows = 1;
      a.tile_pairs = static_cast<int>(tile_pairs_for(segments, n_index, true));
      a.tb_max = static_cast<int>(spread_tiles);
    }
    int rc = launch_bucket<F16>(a, s);  // invalid pairs: zero scales
    if (rc != GRM_HIP_OK) return rc;
    if (segments > 0) {
      switch (mem_dtype) {
        case GRM_HIP_F32: rc = apply_scaled_q<F32>(a, q_dtype, s); break;
        case GRM_HIP_F16: rc = apply_scaled_q<F16>(a, q_dtype, s); break;
        default: rc = apply_scaled_q<BF16>(a, q_dtype, s); break;
      }
      if (rc != GRM_HIP_OK) return rc;
    }
  }
  FuseScaledArgs f;
  f.h = h_online;
  f.rows = reinterpret_cast<const uint16_t*>(rows16);
  f.scales = scales;
  f.all_there = 0;
  f.w = ln_weight;
  f.bias = ln_bias;
  f.out = out;
  f.n_rows = rows;
  f.routes = static_cast<int>(routes);
  f.hidden = static_cast<int>(value_dim);
  f.v_tiles = v_tiles;
  f.eps = eps;
  return fuse_scaled(f, h_dtype, s);
}

namespace {
int gather_apply_bwd_impl(const void* memories, const int64_t* indices, const float* grad_out, float* grad_pairs,
                          void* workspace, int64_t workspace_bytes, int64_t batch, int64_t segments, int64_t n_query,
                          int64_t routes, int64_t hidden_size, int64_t key_dim, int mem_dtype,
                          int32_t* bad_index_count, int token_rows, void* stream) {
  if (batch < 0 || segments < 0 || n_query < 0 || routes < 0 || hidden_size < 0 || key_dim < 1) {
    set_error("gather_apply_bwd: negative size or key_dim < 1");
    return GRM_HIP_EINVAL;
  }
  if (mem_dtype < GRM_HIP_F32 || mem_dtype > GRM_HIP_BF16) {
    set_error("gather_apply_bwd: unsupported memories dtype %d", mem_dtype);
    return GRM_HIP_EUNSUPPORTED;
  }
  const int64_t dkp = key_dim <= 16 ? 16 : key_dim <= 32 ? 32 : key_dim <= 64 ? 64 : 128;
  if (key_dim > 128 || segments > kMaxSegments || hidden_size > (1 << 20) ||
      apply_t_lds(static_cast<int>(hidden_size), static_cast<int>(dkp)) > 160 * 1024) {
    set_error("gather_apply_bwd: needs key_dim <= 128, segments <= %lld and the float32 state in LDS",
              (long long)kMaxSegments);
    return GRM_HIP_EUNSUPPORTED;
  }
  const int64_t n_index = n_query * routes;
  if (batch == 0 || n_index == 0 || key_dim == 0) return GRM_HIP_OK;
  if (n_index > INT32_MAX || batch > 65535 || tiles_max(segments, n_index) > UINT32_MAX) {
    set_error("gather_apply_bwd: sizes exceed one launch");
    return GRM_HIP_EINVAL;
  }
  if (indices == nullptr || grad_pairs == nullptr || (hidden_size > 0 && grad_out == nullptr) ||
      (segments > 0 && memories == nullptr)) {
    set_error("gather_apply_bwd: null pointer");
    return GRM_HIP_EINVAL;
  }
  const int64_t need = grm_hip_gather_apply_workspace(batch, segments, n_index);
  if (workspace == nullptr || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(grad_pairs) % 16 != 0) {
    set_error("gather_apply_bwd: workspace of %lld bytes and 16-byte aligned buffers required", (long long)need);
    return GRM_HIP_EINVAL;
  }
  RetrieveArgs a;
  init_retrieve_args(a, memories, indices, nullptr, grad_pairs, workspace, batch, segments, n_query, routes, n_index,
                     hidden_size, key_dim, bad_index_count);
  a.out_row = static_cast<int>(key_dim);  // invalid pairs: zero gradient rows
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = launch_bucket<F32>(a, s);
  if (rc != GRM_HIP_OK || segments == 0) return rc;
  if (hidden_size == 0) {
    set_error("gather_apply_bwd: value_dim 0 with valid pairs");
    return GRM_HIP_EUNSUPPORTED;
  }
  switch (mem_dtype) {
    case GRM_HIP_F32: return dispatch_apply_t<F32>(a, grad_out, grad_pairs, token_rows, s);
    case GRM_HIP_F16: return dispatch_apply_t<F16>(a, grad_out, grad_pairs, token_rows, s);
    default: return dispatch_apply_t<BF16>(a, grad_out, grad_pairs, token_rows, s);
  }
}
}  // namespace

extern "C" int grm_hip_gather_apply_bwd_queries(const void* memories, const int64_t* indices, const float* grad_out,
                                                float* grad_pairs, void* workspace, int64_t workspace_bytes,
                                                int64_t batch, int64_t segments, int64_t n_query, int64_t routes,
                                                int64_t hidden_size, int64_t key_dim, int mem_dtype,
                                                int32_t* bad_index_count, void* stream) {
  return gather_apply_bwd_impl(memories, indices, grad_out, grad_pairs, workspace, workspace_bytes, batch, segments,
                               n_query, routes, hidden_size, key_dim, mem_dtype, bad_index_count, 0, stream);
}

extern "C" int grm_hip_gather_apply_bwd_tokens(const void* memories, const int64_t* indices, const float* grad_tokens,
                                               float* grad_pairs, void* workspace, int64_t workspace_bytes,
                                               int64_t batch, int64_t segments, int64_t n_query, int64_t routes,
                                               int64_t hidden_size, int64_t key_dim, int mem_dtype,
                                               int32_t* bad_index_count, void* stream) {
  return gather_apply_bwd_impl(memories, indices, grad_tokens, grad_pairs, workspace, workspace_bytes, batch, segments,
                               n_query, routes, hidden_size, key_dim, mem_dtype, bad_index_count, 1, stream);
}
