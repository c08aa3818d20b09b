// Gradient of the chunked linear-memory update + query application in float32
// arithmetic, gfx950: float32 inputs, and 16-bit inputs that the 16-bit MFMA
// kernels of chunk_bwd.hip do not take (odd widths, unaligned rows, key_dim
// above 128).
//
// Adjoint of  M_t = decay M_{t-1} + c v_t k_t^T,  h_t = M_t q_t   (c = (1-decay)/sqrt(d_k))
// (reference grm/csrc/chunk_update.cu:137-278 and :588-716; CPU autograd in
// grm_cuda.cpp:92-126).  Per 64-token chunk of L tokens, from the state M at its
// start and the adjoint G at its end, with D[i][j] = decay^{i-j} (j <= i),
// P = c (Q K^T) o D and dS = c (dH V^T) o D:
//   dQ = decay^{i+1} dH M + dS K
//   dK = dS^T Q + c decay^{L-1-j} V G
//   dV = P^T dH + c decay^{L-1-j} K G^T
//   G at the chunk's start = decay^L G + dH^T diag(decay^{i+1}) Q
// Only the last line carries from chunk to chunk, and its second term does not
// depend on G.  So three launches, each parallel over chunks or elements:
//   bwd_outer_kernel  dH^T diag(decay^{i+1}) Q of every chunk
//   bwd_carry_kernel  the recurrence over chunks, one thread per state element
//   bwd_chunk_kernel  everything else, one workgroup per (sequence, chunk, share
//                     of the value tiles), on float32 MFMA
// With few chunks the value tiles of one chunk are shared by several workgroups
// (`splits`), whose dQ and dK are partial sums that split_sum_kernel adds in order.
// A handful of tokens goes one by one instead (bwd_tokens_kernel, few_tokens).
//
// What bounds it: float32 MFMA (16x16x4, 256 FLOP per CU and clock).  Every
// operand comes from LDS as 16 bytes of a row or as four single elements of a
// column, 64 bytes per clock and CU at most, half of what LDS gives; row strides
// of 4 mod 64 elements keep both forms free of bank conflicts.
//
// Measured, forward and backward of 4 x 2000 float32 tokens, key_dim 64, value_dim
// 512: 9.59 ms with a kernel that swept the tokens one by one (16 value rows per
// wave, 128 waves on the chip), 120 us with these; error of the gradients against
// 64 bits 7.1e-7 before, 2.6e-7 now.
#include <stdint.h>

#include <algorithm>

#include "chunk_bwd.h"
#include "f32_tiles.h"
#include "grm_hip.h"
#include "grm_hip_common.h"

namespace grmhip {
namespace {

constexpr int GNT = 256;          // threads per workgroup
constexpr int GVS = kGenDv + 4;   // LDS row stride of the V and dH tiles
constexpr int GPS = BCT + 4;      // LDS row stride of P and dS
constexpr int OUTER_V = 64;       // value rows per bwd_outer_kernel workgroup

// dH^T diag(decay^{i+1}) Q of one chunk: workgroup (sequence, chunk, 64 value
// rows), wave w rows [16w, +16), every key column.  Operands straight from
// global memory (64-byte row pieces per 16 lanes, each used once per wave).
// One chunk (n_chunks == 1): grad_memory itself, decay^L grad_memory_out added.
template <class E, int DKP>
__global__ __launch_bounds__(GNT) void bwd_outer_kernel(const BwdGenArgs a) {
  using raw = typename ET<E>::raw;
  constexpr int ES = static_cast<int>(sizeof(raw));
  constexpr int KT = DKP / 16;
  __shared__ float pw[BCT + 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dk = a.dk, dv = a.dv;
  const int vtiles = (dv + OUTER_V - 1) / OUTER_V;
  const int vt = static_cast<int>(blockIdx.x % static_cast<unsigned>(vtiles));
  const int64_t bc = blockIdx.x / static_cast<unsigned>(vtiles);
  const int ch = static_cast<int>(bc % a.n_chunks);
  const int64_t b = bc / a.n_chunks;
  const int64_t t0 = static_cast<int64_t>(ch) * BCT;
  const int L = ch == a.n_chunks - 1 ? static_cast<int>(a.T - t0) : BCT;
  if (tid <= BCT) pw[tid] = a.pw[tid];
  __syncthreads();
  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc(static_cast<const raw*>(a.queries) + (b * a.T + t0) * dk, static_cast<uint32_t>(L * dk * ES));
  const __amdgpu_buffer_rsrc_t rh =
      make_rsrc(static_cast<const raw*>(a.dh) + (b * a.T + t0) * dv, static_cast<uint32_t>(L * dv * ES));
  const int v = vt * OUTER_V + 16 * w + n;
  float h[4][4];
#pragma unroll
  for (int ib = 0; ib < 4; ++ib)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = 16 * ib + 4 * g + s;
      h[ib][s] = ET<E>::to_f(buf_load1<E>(rh, v < dv ? (i * dv + v) * ES : kBufOOB));
    }
  f32x4 acc[KT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    const int k = 16 * kt + n;
    float q[4][4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        q[ib][s] = ET<E>::to_f(buf_load1<E>(rq, k < dk ? ((16 * ib + 4 * g + s) * dk + k) * ES : kBufOOB));
    if (kt == 0) {
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int s = 0; s < 4; ++s) h[ib][s] *= pw[16 * ib + 4 * g + s + 1];
    }
    acc[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
      acc[kt] = mfma4(f32x4{q[ib][0], q[ib][1], q[ib][2], q[ib][3]}, f32x4{h[ib][0], h[ib][1], h[ib][2], h[ib][3]},
                      acc[kt]);
  }
  if (v >= dv) return;
  if (a.n_chunks == 1) {
    const float decay_L = pw[L];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * kt + 4 * g + r;
        if (k >= dk) continue;
        const int64_t i = (b * dv + v) * dk + k;
        st_state<E>(a.dm_out, i, a.dm_f32 != 0, fmaf(decay_L, ld_state<E>(a.dmo, i, a.mem_f32 != 0), acc[kt][r]));
      }
    return;
  }
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(a.gbuf + ((b * a.n_chunks + ch) * dv + vt * OUTER_V) * dk,
                                              static_cast<uint32_t>(min(OUTER_V, dv - vt * OUTER_V) * dk * 4));
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    const int k = 16 * kt + 4 * g;
    out4<F32>(ro, (16 * w + n) * dk + k, dk - k, a.vec_k != 0, acc[kt]);
  }
}

// Slot ch := decay^{L_ch} G + slot ch, G the value of slot ch + 1 (grad_memory_out
// for the last chunk): slot ch then holds the adjoint at chunk ch's start, and
// chunk 0's goes to grad_memory.  One thread per state element, eight loads ahead.
template <class E>
__global__ __launch_bounds__(GNT) void bwd_carry_kernel(const BwdGenArgs a) {
  constexpr int AHEAD = 8;
  const int64_t plane = static_cast<int64_t>(a.dv) * a.dk;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * GNT + threadIdx.x;
  if (i >= a.batch * plane) return;
  const int64_t b = i / plane;
  float* slot = a.gbuf + b * a.n_chunks * plane + (i - b * plane);
  float x = ld_state<E>(a.dmo, i, a.mem_f32 != 0);
  const float decay_c = a.pw[BCT];
  const float decay_last = a.pw[static_cast<int>(a.T - static_cast<int64_t>(a.n_chunks - 1) * BCT)];
  float buf[AHEAD];
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) {
    const int ch = a.n_chunks - 1 - j;
    buf[j] = ch >= 0 ? slot[ch * plane] : 0.f;
  }
  for (int top = a.n_chunks - 1; top >= 0; top -= AHEAD) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const int ch = top - j;
      if (ch < 0) break;
      x = fmaf(ch == a.n_chunks - 1 ? decay_last : decay_c, x, buf[j]);
      if (ch > 0) slot[ch * plane] = x;
      const int next = ch - AHEAD;
      buf[j] = next >= 0 ? slot[next * plane] : 0.f;
    }
  }
  st_state<E>(a.dm_out, i, a.dm_f32 != 0, x);
}

// grad_memory from float32 scratch, where it takes the place of an input that
// bwd_chunk_kernel reads.
template <class E>
__global__ __launch_bounds__(GNT) void bwd_state_copy_kernel(const float* from, void* to, int64_t n, int f32) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * GNT + threadIdx.x;
  if (i < n) st_state<E>(to, i, f32 != 0, from[i]);
}

// A few tokens, one by one.  One wave per sequence and 16 value rows, lanes hold the key
// columns in steps of 64: forward over the tokens for M_t and dQ, backward for G_t, dK and
// dV (a reduction over the keys by a 16-value transposing butterfly, 17 shuffles per
// token).  dQ and dK of the 16 rows are partial sums, [batch, value tiles, T, dk].  Bound by
// the latency of each token's loads.
constexpr int TOK_ROWS = 16;
template <class E, int KR>
__global__ __launch_bounds__(64) void bwd_tokens_kernel(const BwdGenArgs a) {
  using raw = typename ET<E>::raw;
  constexpr int RB = TOK_ROWS;
  const int lane = threadIdx.x;
  const int64_t b = blockIdx.x / static_cast<unsigned>(a.splits);
  const int tile = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.splits));
  const int v0 = tile * RB;
  const int dk = a.dk, dv = a.dv, T = static_cast<int>(a.T);
  const float lam = a.pw[1], c = a.c;
  const bool f32m = a.mem_f32 != 0;
  const raw* keys = static_cast<const raw*>(a.keys) + b * T * dk;
  const raw* queries = static_cast<const raw*>(a.queries) + b * T * dk;
  const raw* values = static_cast<const raw*>(a.values) + b * T * dv;
  const raw* dhp = static_cast<const raw*>(a.dh) + b * T * dv;
  const int64_t part = (b * a.splits + tile) * static_cast<int64_t>(T) * dk;
  float M[RB][KR], G[RB][KR];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int e = 0; e < KR; ++e) {
      const int v = v0 + r, k = lane + 64 * e;
      const bool in = v < dv && k < dk;
      const int64_t i = (b * dv + v) * dk + k;
      M[r][e] = in ? ld_state<E>(a.memory, i, f32m) : 0.f;
      G[r][e] = in ? ld_state<E>(a.dmo, i, f32m) : 0.f;
    }
  for (int t = 0; t < T; ++t) {
    float kt[KR], dq[KR];
#pragma unroll
    for (int e = 0; e < KR; ++e) {
      const int k = lane + 64 * e;
      kt[e] = k < dk ? ET<E>::to_f(keys[t * dk + k]) : 0.f;
      dq[e] = 0.f;
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int v = v0 + r;
      const float cv = c * (v < dv ? ET<E>::to_f(values[static_cast<int64_t>(t) * dv + v]) : 0.f);
      const float dh = v < dv ? ET<E>::to_f(dhp[static_cast<int64_t>(t) * dv + v]) : 0.f;
#pragma unroll
      for (int e = 0; e < KR; ++e) {
        M[r][e] = fmaf(M[r][e], lam, cv * kt[e]);
        dq[e] = fmaf(dh, M[r][e], dq[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < KR; ++e)
      if (lane + 64 * e < dk) a.part_q[part + t * dk + lane + 64 * e] = dq[e];
  }
  for (int t = T - 1; t >= 0; --t) {
    float kt[KR], qt[KR], dkt[KR], dvp[RB];
#pragma unroll
    for (int e = 0; e < KR; ++e) {
      const int k = lane + 64 * e;
      kt[e] = k < dk ? ET<E>::to_f(keys[t * dk + k]) : 0.f;
      qt[e] = k < dk ? ET<E>::to_f(queries[t * dk + k]) : 0.f;
      dkt[e] = 0.f;
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int v = v0 + r;
      const float vv = v < dv ? ET<E>::to_f(values[static_cast<int64_t>(t) * dv + v]) : 0.f;
      const float dh = v < dv ? ET<E>::to_f(dhp[static_cast<int64_t>(t) * dv + v]) : 0.f;
      dvp[r] = 0.f;
#pragma unroll
      for (int e = 0; e < KR; ++e) {
        G[r][e] = fmaf(dh, qt[e], t == T - 1 ? G[r][e] : G[r][e] * lam);
        dkt[e] = fmaf(G[r][e], vv, dkt[e]);
        dvp[r] = fmaf(G[r][e], kt[e], dvp[r]);
      }
    }
#pragma unroll
    for (int e = 0; e < KR; ++e)
      if (lane + 64 * e < dk) a.part_k[part + t * dk + lane + 64 * e] = c * dkt[e];
    // 16 row sums over 64 lanes: halve the value count per exchange.
#pragma unroll
    for (int half = RB / 2, d = 32; half >= 1; half >>= 1, d >>= 1) {
      const bool up = (lane & d) != 0;
#pragma unroll
      for (int i = 0; i < half; ++i) {
        const float send = up ? dvp[i] : dvp[i + half];
        const float keep = up ? dvp[i + half] : dvp[i];
        dvp[i] = keep + __shfl_xor(send, d, 64);
      }
    }
    float tot = dvp[0];
    tot += __shfl_xor(tot, 2, 64);
    tot += __shfl_xor(tot, 1, 64);
    const int v = v0 + ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 2) & 1);
    if ((lane & 3) == 0 && v < dv)
      static_cast<raw*>(a.dv_out)[(b * T + t) * dv + v] = ET<E>::from_f(c * tot);
  }
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int e = 0; e < KR; ++e) {
      const int v = v0 + r, k = lane + 64 * e;
      if (v < dv && k < dk) st_state<E>(a.dm_out, (b * dv + v) * dk + k, f32m, G[r][e] * lam);
    }
}

template <class E, int DKP>
struct GenShape {
  using raw = typename ET<E>::raw;
  static constexpr int KS = DKP + 4;  // LDS row stride of K, Q (input type) and of M, G (float32)
  static constexpr int KT = DKP / 16;
  static constexpr int KQ_LOADS = BCT * DKP / GNT;
  static constexpr int V_LOADS = BCT * kGenDv / GNT;
  static constexpr int M_LOADS = kGenDv * DKP / GNT;
  static constexpr size_t kq_bytes = 2ull * BCT * KS * sizeof(raw);
  static constexpr size_t vh_bytes = 2ull * BCT * GVS * sizeof(raw);
  static constexpr size_t mg_bytes = 2ull * kGenDv * KS * 4;
  static constexpr size_t p_bytes = static_cast<size_t>(BCT) * GPS * 4;
  // P (before the first value tile) and dS (after the last) share the value tiles' region.
  static constexpr size_t tile_bytes = vh_bytes + mg_bytes > p_bytes ? vh_bytes + mg_bytes : p_bytes;
  static constexpr size_t lds_bytes = kq_bytes + tile_bytes + (BCT + 1) * 4;
  static_assert(lds_bytes <= 160 * 1024, "one workgroup's tiles fit the CU");
  static_assert(kq_bytes % 16 == 0 && vh_bytes % 16 == 0 && tile_bytes % 16 == 0, "16-byte regions");
};

// The gradients of one chunk from its starting state and the adjoint at its end,
// over value tiles [split * tiles_per_split, +tiles_per_split).  Wave w owns tokens
// [16w, +16) of every product; lane (g, n) of an accumulator holds four
// consecutive key (or value) columns 4g + r of token n.
template <class E, int DKP>
__global__ __launch_bounds__(GNT) void bwd_chunk_kernel(const BwdGenArgs a) {
  using S = GenShape<E, DKP>;
  using raw = typename ET<E>::raw;
  constexpr int ES = static_cast<int>(sizeof(raw));
  constexpr int KS = S::KS, KT = S::KT;
  extern __shared__ __align__(16) unsigned char smem[];
  raw* Ks = reinterpret_cast<raw*>(smem);  // [BCT][KS]
  raw* Qs = Ks + BCT * KS;                 // [BCT][KS]
  unsigned char* tile = smem + S::kq_bytes;
  raw* Vs = reinterpret_cast<raw*>(tile);  // [BCT][GVS] value tile columns
  raw* Hs = Vs + BCT * GVS;                // [BCT][GVS] grad_hidden tile columns
  float* Ms = reinterpret_cast<float*>(tile + S::vh_bytes);  // [kGenDv][KS] the chunk's starting state
  float* Gs = Ms + kGenDv * KS;                              // [kGenDv][KS] adjoint at the chunk's end
  float* Ps = reinterpret_cast<float*>(tile);                // [BCT][GPS] P, then dS
  float* pw = reinterpret_cast<float*>(tile + S::tile_bytes);

  const int tid = threadIdx.x;
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.splits));
  const int64_t bc = blockIdx.x / static_cast<unsigned>(a.splits);
  const int ch = static_cast<int>(bc % a.n_chunks);
  const int64_t b = bc / a.n_chunks;
  const int dk = a.dk, dv = a.dv;
  const int64_t t0 = static_cast<int64_t>(ch) * BCT;
  const int L = ch == a.n_chunks - 1 ? static_cast<int>(a.T - t0) : BCT;
  const float c = a.c;
  const bool f32m = a.mem_f32 != 0;
  const int64_t mem_b = f32m ? 4 : ES;
  const int vt_begin = split * a.tiles_per_split;
  const int vt_end = min(vt_begin + a.tiles_per_split, (dv + kGenDv - 1) / kGenDv);

  if (tid <= BCT) pw[tid] = a.pw[tid];
  {
    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(static_cast<const raw*>(a.keys) + (b * a.T + t0) * dk, static_cast<uint32_t>(L * dk * ES));
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(static_cast<const raw*>(a.queries) + (b * a.T + t0) * dk, static_cast<uint32_t>(L * dk * ES));
    constexpr int STEP = S::KQ_LOADS < 16 ? S::KQ_LOADS : 16;
#pragma unroll 1
    for (int u0 = 0; u0 < S::KQ_LOADS; u0 += STEP) {
      raw kx[STEP], qx[STEP];
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + GNT * (u0 + u), row = l / DKP, col = l % DKP;
        const int off = col < dk ? (row * dk + col) * ES : kBufOOB;
        kx[u] = buf_load1<E>(rk, off);
        qx[u] = buf_load1<E>(rq, off);
      }
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + GNT * (u0 + u), row = l / DKP, col = l % DKP;
        Ks[row * KS + col] = kx[u];
        Qs[row * KS + col] = qx[u];
      }
    }
  }

  const unsigned char* msrc =
      ch == 0 ? static_cast<const unsigned char*>(a.memory) + b * dv * dk * mem_b
              : reinterpret_cast<const unsigned char*>(a.states + (b * a.n_chunks + ch - 1) * dv * dk);
  const unsigned char* gsrc =
      ch == a.n_chunks - 1 ? static_cast<const unsigned char*>(a.dmo) + b * dv * dk * mem_b
                           : reinterpret_cast<const unsigned char*>(a.gbuf + (b * a.n_chunks + ch + 1) * dv * dk);
  const bool m32 = ch != 0 || f32m, g32 = ch != a.n_chunks - 1 || f32m;
  const __amdgpu_buffer_rsrc_t rv =
      make_rsrc(static_cast<const raw*>(a.values) + (b * a.T + t0) * dv, static_cast<uint32_t>(L * dv * ES));
  const __amdgpu_buffer_rsrc_t rh =
      make_rsrc(static_cast<const raw*>(a.dh) + (b * a.T + t0) * dv, static_cast<uint32_t>(L * dv * ES));
  struct Stage {
    raw v[S::V_LOADS], h[S::V_LOADS];
    float m[S::M_LOADS], gg[S::M_LOADS];
  };
  auto load_vtile = [&](int vt, Stage& sg) {
    const int v0 = vt * kGenDv;
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + GNT * u, row = l / kGenDv, col = v0 + l % kGenDv;
      const int off = col < dv ? (row * dv + col) * ES : kBufOOB;
      sg.v[u] = buf_load1<E>(rv, off);
      sg.h[u] = buf_load1<E>(rh, off);
    }
    const int rows = min(kGenDv, dv - v0);
    const int mb = m32 ? 4 : ES, gb = g32 ? 4 : ES;
    const __amdgpu_buffer_rsrc_t rm =
        make_rsrc(msrc + static_cast<int64_t>(v0) * dk * mb, static_cast<uint32_t>(rows * dk * mb));
    const __amdgpu_buffer_rsrc_t rg =
        make_rsrc(gsrc + static_cast<int64_t>(v0) * dk * gb, static_cast<uint32_t>(rows * dk * gb));
#pragma unroll
    for (int u = 0; u < S::M_LOADS; ++u) {
      const int l = tid + GNT * u, row = l / DKP, col = l % DKP;
      sg.m[u] = ld_mem(rm, row * dk + col, m32, col < dk, E());
      sg.gg[u] = ld_mem(rg, row * dk + col, g32, col < dk, E());
    }
  };
  auto store_vtile = [&](const Stage& sg) {
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + GNT * u, o = (l / kGenDv) * GVS + l % kGenDv;
      Vs[o] = sg.v[u];
      Hs[o] = sg.h[u];
    }
#pragma unroll
    for (int u = 0; u < S::M_LOADS; ++u) {
      const int l = tid + GNT * u, o = (l / DKP) * KS + l % DKP;
      Ms[o] = sg.m[u];
      Gs[o] = sg.gg[u];
    }
  };
  Stage stage;
  load_vtile(vt_begin, stage);
  __syncthreads();  // K, Q, pw

  // c decay^{i-j} x for this lane's row i = 16w + n and keys j = 16 jb + 4g + r, zero right of the diagonal
  const int jrow = 16 * w + n;
  auto causal4 = [&](int jb, f32x4 x) {
    f32x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * jb + 4 * g + r;
      y[r] = j <= jrow ? x[r] * (c * pw[max(jrow - j, 0)]) : 0.f;
    }
    return y;
  };
  const float sq = pw[jrow + 1];
  const float wl = (jrow < L) ? c * pw[max(L - 1 - jrow, 0)] : 0.f;

  // ---- P rows of query block w, then this wave's columns of P
  f32x4 pT[4];
  {
    f32x4 s[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) s[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int kk = 0; kk < KT; ++kk) {
      const f32x4 qf = lds_row4<E>(Qs + jrow * KS + 16 * kk + 4 * g);
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= w) s[jb] = mfma4(lds_row4<E>(Ks + (16 * jb + n) * KS + 16 * kk + 4 * g), qf, s[jb]);
    }
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      *reinterpret_cast<float4*>(Ps + jrow * GPS + 16 * jb + 4 * g) =
          __builtin_bit_cast(float4, causal4(jb, s[jb]));
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) pT[ib] = lds_col4<F32>(Ps + (16 * ib + 4 * g) * GPS + jrow, GPS);
    __syncthreads();  // P read: the region takes the value tiles
  }

  // NaN once a result is not finite
  float check = 0.f;
  auto finite = [&](f32x4 x) {
#pragma unroll
    for (int r = 0; r < 4; ++r) check = fmaf(x[r], 0.f, check);
  };
  f32x4 dsacc[4], dq[KT], dkk[KT];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) dsacc[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) dq[kt] = dkk[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const __amdgpu_buffer_rsrc_t rdv =
      make_rsrc(static_cast<raw*>(a.dv_out) + (b * a.T + t0) * dv, static_cast<uint32_t>(L * dv * ES));
  for (int vt = vt_begin; vt < vt_end; ++vt) {
    store_vtile(stage);
    if (vt + 1 < vt_end) load_vtile(vt + 1, stage);
    __syncthreads();  // value tile in LDS
#pragma unroll
    for (int cc = 0; cc < kGenDv / 16; ++cc) {
      const f32x4 hf = lds_row4<E>(Hs + jrow * GVS + 16 * cc + 4 * g);
      const f32x4 vf = lds_row4<E>(Vs + jrow * GVS + 16 * cc + 4 * g);
      // dS rows of block w
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= w) dsacc[jb] = mfma4(lds_row4<E>(Vs + (16 * jb + n) * GVS + 16 * cc + 4 * g), hf, dsacc[jb]);
      // dQ (sum_v dH[i][v] M[v][k]) and dK (sum_v G[v][k] V[j][v])
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const int o = (16 * cc + 4 * g) * KS + 16 * kt + n;
        dq[kt] = mfma4(lds_col4<F32>(Ms + o, KS), hf, dq[kt]);
        dkk[kt] = mfma4(lds_col4<F32>(Gs + o, KS), vf, dkk[kt]);
      }
    }
    // dV rows of block w: c decay^{L-1-j} sum_k G[v][k] K[j][k] + sum_i dH[i][v] P[i][j]
    f32x4 dvv[kGenDv / 16];
#pragma unroll
    for (int vb = 0; vb < kGenDv / 16; ++vb) dvv[vb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int kk = 0; kk < KT; ++kk) {
      const f32x4 kf = lds_row4<E>(Ks + jrow * KS + 16 * kk + 4 * g);
#pragma unroll
      for (int vb = 0; vb < kGenDv / 16; ++vb)
        dvv[vb] = mfma4(lds_row4<F32>(Gs + (16 * vb + n) * KS + 16 * kk + 4 * g), kf, dvv[vb]);
    }
#pragma unroll
    for (int vb = 0; vb < kGenDv / 16; ++vb) {
      f32x4 acc = dvv[vb] * wl;
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
        if (ib >= w) acc = mfma4(lds_col4<E>(Hs + (16 * ib + 4 * g) * GVS + 16 * vb + n, GVS), pT[ib], acc);
      finite(acc);
      const int v = vt * kGenDv + 16 * vb + 4 * g;
      out4<E>(rdv, jrow * dv + v, dv - v, a.vec_v != 0, acc);
    }
    __syncthreads();  // every read of this tile done
  }

  // ---- dS complete.  dQ takes this wave's rows from registers (the accumulator
  // layout is the operand layout), dK this wave's columns through LDS.
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) {
    dsacc[jb] = causal4(jb, dsacc[jb]);
    *reinterpret_cast<float4*>(Ps + jrow * GPS + 16 * jb + 4 * g) = __builtin_bit_cast(float4, dsacc[jb]);
  }
  __syncthreads();
  f32x4 dsT[4];
#pragma unroll
  for (int ib = 0; ib < 4; ++ib) dsT[ib] = lds_col4<F32>(Ps + (16 * ib + 4 * g) * GPS + jrow, GPS);
  const bool partial = a.splits > 1;
  const int64_t prow = ((b * a.splits + split) * a.T + t0) * dk;
  const __amdgpu_buffer_rsrc_t rqo =
      partial ? make_rsrc(a.part_q + prow, static_cast<uint32_t>(L * dk * 4))
              : make_rsrc(static_cast<raw*>(a.dq_out) + (b * a.T + t0) * dk, static_cast<uint32_t>(L * dk * ES));
  const __amdgpu_buffer_rsrc_t rko =
      partial ? make_rsrc(a.part_k + prow, static_cast<uint32_t>(L * dk * 4))
              : make_rsrc(static_cast<raw*>(a.dk_out) + (b * a.T + t0) * dk, static_cast<uint32_t>(L * dk * ES));
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    f32x4 aq = dq[kt] * sq, ak = dkk[kt] * wl;
#pragma unroll
    for (int xb = 0; xb < 4; ++xb) {
      const int o = (16 * xb + 4 * g) * KS + 16 * kt + n;
      if (xb <= w) aq = mfma4(lds_col4<E>(Ks + o, KS), dsacc[xb], aq);
      if (xb >= w) ak = mfma4(lds_col4<E>(Qs + o, KS), dsT[xb], ak);
    }
    finite(aq);
    finite(ak);
    const int k = 16 * kt + 4 * g;
    if (partial) {
      out4<F32>(rqo, jrow * dk + k, dk - k, a.vec_k != 0, aq);
      out4<F32>(rko, jrow * dk + k, dk - k, a.vec_k != 0, ak);
    } else {
      out4<E>(rqo, jrow * dk + k, dk - k, a.vec_k != 0, aq);
      out4<E>(rko, jrow * dk + k, dk - k, a.vec_k != 0, ak);
    }
  }
  if (a.exact == 0 || !__any(check != check)) return;

  // ---- Some result of this wave's tokens is not finite.  The products above multiply the
  // zeros above the diagonal too, and zero times an infinity or NaN is NaN: a token's would
  // reach the gradients of its whole 16-token block.  The wave's rows once more, one product
  // at a time and only those that belong to a gradient.  Lane (g, n): token 16w + n, columns
  // 8g .. 8g + 7 of every 32.  dQ and dK first: dS is in LDS.
  const __amdgpu_buffer_rsrc_t rm = make_rsrc(msrc, static_cast<uint32_t>(dv * dk * (m32 ? 4 : ES)));
  const __amdgpu_buffer_rsrc_t rg = make_rsrc(gsrc, static_cast<uint32_t>(dv * dk * (g32 ? 4 : ES)));
  const int v_begin = vt_begin * kGenDv, v_end = min(vt_end * kGenDv, dv);
#pragma unroll 1
  for (int k0 = 8 * g; k0 < DKP; k0 += 32) {
    float aq[8], ak[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) aq[e] = ak[e] = 0.f;
#pragma unroll 1
    for (int v = v_begin; v < v_end; ++v) {
      const float hx = ET<E>::to_f(buf_load1<E>(rh, (jrow * dv + v) * ES));  // zero from token L on
      const float vx = ET<E>::to_f(buf_load1<E>(rv, (jrow * dv + v) * ES));
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        aq[e] = fmaf(hx, ld_mem(rm, v * dk + k0 + e, m32, k0 + e < dk, E()), aq[e]);
        ak[e] = fmaf(vx, ld_mem(rg, v * dk + k0 + e, g32, k0 + e < dk, E()), ak[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      aq[e] *= sq;
      ak[e] *= wl;
    }
#pragma unroll 1
    for (int x = 0; x < L; ++x) {
      const float dsq = Ps[jrow * GPS + x], dsk = Ps[x * GPS + jrow];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (x <= jrow) aq[e] = fmaf(dsq, ET<E>::to_f(Ks[x * KS + k0 + e]), aq[e]);
        if (x >= jrow) ak[e] = fmaf(dsk, ET<E>::to_f(Qs[x * KS + k0 + e]), ak[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int off = jrow < L && k0 + e < dk ? jrow * dk + k0 + e : -1;
      if (partial) {
        buf_store1<F32>(rqo, off >= 0 ? off * 4 : kBufOOB, aq[e]);
        buf_store1<F32>(rko, off >= 0 ? off * 4 : kBufOOB, ak[e]);
      } else {
        buf_store1<E>(rqo, off >= 0 ? off * ES : kBufOOB, aq[e]);
        buf_store1<E>(rko, off >= 0 ? off * ES : kBufOOB, ak[e]);
      }
    }
  }
#pragma unroll 1
  for (int v0 = v_begin + 8 * g; v0 < v_end; v0 += 32) {
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll 1
    for (int k = 0; k < dk; ++k) {
      const float kx = ET<E>::to_f(Ks[jrow * KS + k]);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(ld_mem(rg, (v0 + e) * dk + k, g32, v0 + e < dv, E()), kx, acc[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= wl;
#pragma unroll 1
    for (int i = jrow; i < L; ++i) {
      float p = 0.f;
#pragma unroll 1
      for (int k = 0; k < dk; ++k) p = fmaf(ET<E>::to_f(Qs[i * KS + k]), ET<E>::to_f(Ks[jrow * KS + k]), p);
      p *= c * pw[i - jrow];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        acc[e] = fmaf(ET<E>::to_f(buf_load1<E>(rh, v0 + e < dv ? (i * dv + v0 + e) * ES : kBufOOB)), p, acc[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      buf_store1<E>(rdv, jrow < L && v0 + e < dv ? (jrow * dv + v0 + e) * ES : kBufOOB, acc[e]);
  }
}

// out[b, t, k] = sum over splits of part[b, split, t, k], splits in order;
// blockIdx.y 0: grad_keys, 1: grad_queries.
template <class E>
__global__ __launch_bounds__(GNT) void split_sum_kernel(const BwdGenArgs a) {
  const float* part = blockIdx.y == 0 ? a.part_k : a.part_q;
  void* out = blockIdx.y == 0 ? a.dk_out : a.dq_out;
  const int64_t plane = a.T * a.dk, total = a.batch * plane;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * GNT + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * GNT) {
    const int64_t b = i / plane;
    const float* p = part + b * a.splits * plane + (i - b * plane);
    float s = p[0];
    for (int x = 1; x < a.splits; ++x) s += p[x * plane];
    static_cast<typename ET<E>::raw*>(out)[i] = ET<E>::from_f(s);
  }
}

template <class E>
int launch_split_sum(const BwdGenArgs& a, hipStream_t s) {
  const int64_t want = (a.batch * a.T * a.dk + GNT - 1) / GNT;
  hipLaunchKernelGGL(split_sum_kernel<E>, dim3(static_cast<unsigned>(std::min<int64_t>(want, 4096)), 2), dim3(GNT), 0,
                     s, a);
  return check_launch("chunk_update_bwd(split sum)");
}

// copy_to: grad_memory where a.dm_out is scratch, else NULL.
template <class E, int DKP>
int launch_gen(const BwdGenArgs& a, void* copy_to, hipStream_t s) {
  using S = GenShape<E, DKP>;
  if (S::lds_bytes > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_chunk_kernel<E, DKP>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(S::lds_bytes));
    if (e != hipSuccess) {
      set_error("chunk_update_bwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
  }
  const int64_t bc = a.batch * a.n_chunks;
  const int64_t n = a.batch * a.dv * a.dk;
  const dim3 state_grid(static_cast<unsigned>((n + GNT - 1) / GNT));
  hipLaunchKernelGGL((bwd_outer_kernel<E, DKP>), dim3(static_cast<unsigned>(bc * ((a.dv + OUTER_V - 1) / OUTER_V))),
                     dim3(GNT), 0, s, a);
  int rc = check_launch("chunk_update_bwd(outer)");
  if (rc != GRM_HIP_OK) return rc;
  if (a.n_chunks > 1) {
    hipLaunchKernelGGL(bwd_carry_kernel<E>, state_grid, dim3(GNT), 0, s, a);
    rc = check_launch("chunk_update_bwd(carry)");
    if (rc != GRM_HIP_OK) return rc;
  }
  hipLaunchKernelGGL((bwd_chunk_kernel<E, DKP>), dim3(static_cast<unsigned>(bc * a.splits)), dim3(GNT), S::lds_bytes, s,
                     a);
  rc = check_launch("chunk_update_bwd(gradients)");
  if (rc != GRM_HIP_OK) return rc;
  if (copy_to != nullptr) {
    hipLaunchKernelGGL(bwd_state_copy_kernel<E>, state_grid, dim3(GNT), 0, s, static_cast<const float*>(a.dm_out),
                       copy_to, n, a.mem_f32);
    rc = check_launch("chunk_update_bwd(state copy)");
    if (rc != GRM_HIP_OK) return rc;
  }
  return a.splits == 1 ? rc : launch_split_sum<E>(a, s);
}

template <class E>
int launch_tokens(const BwdGenArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.batch * a.splits));
  if (a.dk <= 64) hipLaunchKernelGGL((bwd_tokens_kernel<E, 1>), grid, dim3(64), 0, s, a);
  else if (std::is_same_v<E, F32> || a.dk <= 128)
    hipLaunchKernelGGL((bwd_tokens_kernel<E, 2>), grid, dim3(64), 0, s, a);
  else if constexpr (!std::is_same_v<E, F32>)
    hipLaunchKernelGGL((bwd_tokens_kernel<E, 4>), grid, dim3(64), 0, s, a);
  const int rc = check_launch("chunk_update_bwd(tokens)");
  return rc != GRM_HIP_OK ? rc : launch_split_sum<E>(a, s);
}

template <class E>
int launch_gen_width(const BwdGenArgs& a, void* copy_to, hipStream_t s) {
  if (a.dk <= 32) return launch_gen<E, 32>(a, copy_to, s);
  if (a.dk <= 64) return launch_gen<E, 64>(a, copy_to, s);
  if (a.dk <= 128) return launch_gen<E, 128>(a, copy_to, s);
  if constexpr (sizeof(typename ET<E>::raw) == 2) return launch_gen<E, 256>(a, copy_to, s);
  set_error("chunk_update_bwd: key_dim %d exceeds 128 for float32", a.dk);
  return GRM_HIP_EUNSUPPORTED;
}

// Workgroups of one chunk's value tiles: enough for two per CU, at least two tiles each
// (a split repeats the chunk's P and its dS products, worth about one tile's work).
int64_t splits_for(int64_t chunks, int64_t vtiles) {
  return std::max<int64_t>(1, std::min<int64_t>((512 + chunks - 1) / chunks, vtiles / 2));
}

// Token by token where a 64-token chunk is mostly padding: it costs its 20 to 80 us
// whatever T, a token 5 (float32) to 10 us.  Whole call, chunk kernels and token kernel, us:
//   key_dim 64, value_dim 64, 16 sequences, float32: 2 tokens 26 and 22, 3 tokens 26 and 24,
//     4 tokens 26 and 28; float16: 29 and 26, 28 and 34
//   (128, 128), 16 sequences, float32: 1 token 44 and 21, 5 tokens 44 and 40, 6 tokens 44
//     and 45; float16: 3 tokens 47 and 40, 4 tokens 48 and 49; key_dim 200, 5 tokens 82 and 68
//   (128, 128), 256 sequences (more workgroups than the one per CU that its LDS allows),
//     float32: 8 tokens 78 and 67, 12 tokens 79 and 108; float16: 4 tokens 82 and 60
//   up to 32 keys the chunk kernels are at the host's 21 us for any of these
// It also takes the short calls that have no room for grad_memory in scratch.
bool few_tokens(const BwdGenArgs& a, int in_dtype, bool in_place) {
  const bool f32 = in_dtype == GRM_HIP_F32;
  const bool full = a.batch * splits_for(a.batch, (a.dv + kGenDv - 1) / kGenDv) > 256;
  const int most = a.dk <= 32    ? 0
                   : a.dk <= 64  ? (f32 ? 3 : 2)
                   : a.dk <= 128 ? (f32 ? (full ? 8 : 5) : (full ? 4 : 3))
                                 : 5;
  return a.T <= most || (in_place && a.T < 8);
}

}  // namespace

int launch_bwd_gen(BwdGenArgs a, int in_dtype, float* ws, int64_t floats, hipStream_t s) {
  const int64_t state = a.batch * static_cast<int64_t>(a.dv) * a.dk, state_b = state * (a.mem_f32 != 0 ? 4 : 2);
  const bool in_place =
      ranges_overlap(a.dm_out, state_b, a.dmo, state_b) || ranges_overlap(a.dm_out, state_b, a.memory, state_b);
  const int64_t rows = a.batch * a.T * a.dk;
  a.dm_f32 = a.mem_f32;
  if (few_tokens(a, in_dtype, in_place)) {
    a.splits = (a.dv + TOK_ROWS - 1) / TOK_ROWS;
    a.part_k = ws;
    a.part_q = ws + a.splits * rows;
    switch (in_dtype) {
      case GRM_HIP_F32: return launch_tokens<F32>(a, s);
      case GRM_HIP_F16: return launch_tokens<F16>(a, s);
      default: return launch_tokens<BF16>(a, s);
    }
  }
  const int64_t vtiles = (a.dv + kGenDv - 1) / kGenDv;
  int64_t adj = a.n_chunks > 1 ? a.n_chunks * state : 0;
  // grad_memory in the place of grad_memory_out or memory, which bwd_chunk_kernel reads: it
  // goes through scratch behind the adjoints, for which the documented workspace has room
  // from eight tokens on.
  void* copy_to = nullptr;
  if (in_place && adj + state <= floats) {
    copy_to = a.dm_out;
    a.dm_out = ws + adj;
    a.dm_f32 = 1;
    adj += state;
  }
  const int64_t bc = a.batch * a.n_chunks;
  int64_t splits = splits_for(bc, vtiles);  // fewer where their partial sums exceed the workspace
  while (splits > 1 && adj + 2 * splits * rows > floats) --splits;
  const int64_t per = (vtiles + splits - 1) / splits;
  a.tiles_per_split = static_cast<int>(per);
  a.splits = static_cast<int>((vtiles + per - 1) / per);
  if (adj > floats || std::min<int64_t>(a.T, BCT) * a.dv * 4 > INT32_MAX || bc * a.splits > INT32_MAX ||
      bc * ((a.dv + OUTER_V - 1) / OUTER_V) > INT32_MAX || (state + GNT - 1) / GNT > INT32_MAX) {
    set_error("chunk_update_bwd: problem too large for one launch");
    return GRM_HIP_EINVAL;
  }
  // bwd_chunk_kernel may read values and grad_hidden again after it has written gradients.
  a.exact = static_cast<int64_t>(a.dv) * a.dk * 4 <= INT32_MAX;
  const int64_t es = in_dtype == GRM_HIP_F32 ? 4 : 2, kb = rows * es, vb = a.batch * a.T * a.dv * es;
  const void* const outs[] = {a.dq_out, a.dk_out, a.dv_out};
  const int64_t out_b[] = {kb, kb, vb};
  for (int o = 0; o < 3; ++o)
    if (ranges_overlap(outs[o], out_b[o], a.values, vb) || ranges_overlap(outs[o], out_b[o], a.dh, vb)) a.exact = 0;
  a.gbuf = ws;
  a.part_k = ws + adj;
  a.part_q = ws + adj + a.splits * rows;
  switch (in_dtype) {
    case GRM_HIP_F32: return launch_gen_width<F32>(a, copy_to, s);
    case GRM_HIP_F16: return launch_gen_width<F16>(a, copy_to, s);
    default: return launch_gen_width<BF16>(a, copy_to, s);
  }
}

}  // namespace grmhip
