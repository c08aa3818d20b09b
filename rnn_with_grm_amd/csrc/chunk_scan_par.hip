// The chunked scan with its chunks in parallel, gfx950: float32 inputs, and 16-bit
// ones that the 16-bit kernels do not take, where sequences and value tiles alone are
// too few workgroups to fill the chip (maths and layouts: chunk_scan.hip).
//
// Walking a sequence chunk by chunk costs 4-5 us per 64-token chunk (a chain of LDS
// round trips and float32 MFMAs), and the S = Q K^T of a chunk is repeated for every
// 32-column value tile.  Here a workgroup takes one chunk:
//   few chunks (par_direct): one launch (fwd_chunk_kernel<.., true>).  Each
//     workgroup forms the state at its chunk's start itself, by walking the earlier
//     chunks' K and V (no S, no outputs), then its outputs; one more per sequence
//     forms the last state.
//   more chunks: fwd_outer_kernel forms every chunk's own contribution to the state,
//     fwd_carry_kernel carries them over the chunks in place, one thread per state
//     element, and fwd_chunk_kernel<.., false> takes the starting state from there.
//     The slots of that carry are the caller's snapshots when one follows every
//     chunk, else workspace.
// Bound by float32 MFMA (256 FLOP per CU and clock) at large sizes and by the loads'
// latency at small ones.  Measured, float32, with a snapshot every 64 tokens, against the
// walk: 4 x 2000 tokens (key_dim 64, value_dim 512) 52.8 -> 42 us, 8 x 1000 (32, 256) 39 -> 24,
// 2 x 4000 (128, 128) 95 -> 39, 1 x 16000 (64, 128) 69 -> 49; 3 x 1000 bf16 (25, 100) 31 -> 22.
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "chunk_scan.h"
#include "f32_tiles.h"
#include "grm_hip.h"
#include "grm_hip_common.h"

namespace grmhip {
namespace {

constexpr int PNT = 256;
constexpr int PDV = 32;        // value columns per tile
constexpr int PVS = PDV + 4;   // LDS row stride of the V tile

// Workgroups up to which the one-launch form is taken: one per CU (each repeats the
// state of all earlier chunks; float32, 4 chunks: 160 workgroups 20.6 us walked, 15.1 here,
// about the host's own time for the call; 640 workgroups 22.0 walked, 29.8 here).
constexpr int64_t kParDirectWgs = 256;

struct ParArgs {
  ChunkFwdArgs f;
  float* slots;         // [B, n_chunks, dv, dk] state after each chunk (not in the one-launch form)
  int splits;           // workgroups sharing one chunk's value tiles
  int tiles_per_split;
  int vec_k, vec_v;     // rows allow 4-element stores
};

__device__ __forceinline__ int chunk_tokens(const ChunkFwdArgs& f, int ch) {
  return ch == f.n_chunks - 1 ? static_cast<int>(f.seq_len - static_cast<int64_t>(ch) * f.chunk) : f.chunk;
}

// A state tile's 16-key x 16-value blocks over the four waves: wave w owns key tiles
// kt0 + kstep q and value blocks vb0 + i (one of the two where there are only two key tiles).
template <int DKP>
struct ParWidth {
  static constexpr int KT = DKP / 16;
  static constexpr int VBW = KT < 4 ? 1 : 2;    // value blocks per wave
  static constexpr int KSTEP = KT < 4 ? KT : 4;
  static constexpr int KTW = KT / KSTEP;        // key tiles per wave
  __device__ static int kt0(int w) { return w % KSTEP; }
  __device__ static int vb0(int w) { return VBW == 1 ? w / KSTEP : 0; }
};

// The operands of one chunk's contribution K^T (w V) to the state, straight from global
// memory, for the blocks of wave w and the 32 value columns at v0.
template <class E, int DKP>
struct OuterOps {
  using W = ParWidth<DKP>;
  using raw = typename ET<E>::raw;
  static constexpr int ES = static_cast<int>(sizeof(raw));
  raw k[W::KTW][4][4], v[W::VBW][4][4];
  __device__ __forceinline__ void load(const ChunkFwdArgs& f, int64_t b, int ch, int v0, int w, int g, int n) {
    const int dk = f.dk, dv = f.dv, L = chunk_tokens(f, ch);
    const int64_t t0 = b * f.seq_len + static_cast<int64_t>(ch) * f.chunk;
    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(static_cast<const raw*>(f.keys) + t0 * dk, static_cast<uint32_t>(L * dk * ES));
    const __amdgpu_buffer_rsrc_t rv =
        make_rsrc(static_cast<const raw*>(f.values) + t0 * dv, static_cast<uint32_t>(L * dv * ES));
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int j = 16 * ib + 4 * g + s;
#pragma unroll
        for (int q = 0; q < W::KTW; ++q) {
          const int kc = 16 * (W::kt0(w) + W::KSTEP * q) + n;
          k[q][ib][s] = buf_load1<E>(rk, kc < dk ? (j * dk + kc) * ES : kBufOOB);
        }
#pragma unroll
        for (int vb = 0; vb < W::VBW; ++vb) {
          const int vc = v0 + 16 * (W::vb0(w) + vb) + n;
          v[vb][ib][s] = buf_load1<E>(rv, vc < dv ? (j * dv + vc) * ES : kBufOOB);
        }
      }
  }
};

// acc[q][vb] += K^T (w V), w_j = c decay^{L-1-j}; lane (g, n) of a result holds keys
// 16 kt + 4 g + r of value 16 vb + n.
template <class E, int DKP>
__device__ __forceinline__ void outer_mac(const OuterOps<E, DKP>& x, int L, float c, int g, const float* pw,
                                          f32x4 (&acc)[ParWidth<DKP>::KTW][ParWidth<DKP>::VBW]) {
  using W = ParWidth<DKP>;
#pragma unroll
  for (int ib = 0; ib < 4; ++ib) {
    f32x4 wv[W::VBW];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int j = 16 * ib + 4 * g + s;
      const float wj = j < L ? c * pw[max(L - 1 - j, 0)] : 0.f;
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb) wv[vb][s] = ET<E>::to_f(x.v[vb][ib][s]) * wj;
    }
#pragma unroll
    for (int q = 0; q < W::KTW; ++q) {
      f32x4 ka;
#pragma unroll
      for (int s = 0; s < 4; ++s) ka[s] = ET<E>::to_f(x.k[q][ib][s]);
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb) acc[q][vb] = mfma4(ka, wv[vb], acc[q][vb]);
    }
  }
}

// Every chunk's contribution to the state, workgroup (sequence, chunk, 32 value columns).
template <class E, int DKP>
__global__ __launch_bounds__(PNT) void fwd_outer_kernel(const ParArgs a) {
  using W = ParWidth<DKP>;
  __shared__ float pw[PW_N];
  const ChunkFwdArgs& f = a.f;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int vtiles = (f.dv + PDV - 1) / PDV;
  const int v0 = static_cast<int>(blockIdx.x % static_cast<unsigned>(vtiles)) * PDV;
  const int64_t bc = blockIdx.x / static_cast<unsigned>(vtiles);
  const int ch = static_cast<int>(bc % f.n_chunks);
  const int64_t b = bc / f.n_chunks;
  if (tid < PW_N) pw[tid] = f.pw[tid];
  __syncthreads();
  f32x4 acc[W::KTW][W::VBW];
#pragma unroll
  for (int q = 0; q < W::KTW; ++q)
#pragma unroll
    for (int vb = 0; vb < W::VBW; ++vb) acc[q][vb] = f32x4{0.f, 0.f, 0.f, 0.f};
  OuterOps<E, DKP> ops;
  ops.load(f, b, ch, v0, w, g, n);
  outer_mac<E, DKP>(ops, chunk_tokens(f, ch), f.c, g, pw, acc);
  const int rows = min(PDV, f.dv - v0);
  const __amdgpu_buffer_rsrc_t ro =
      make_rsrc(a.slots + ((b * f.n_chunks + ch) * f.dv + v0) * f.dk, static_cast<uint32_t>(rows * f.dk * 4));
#pragma unroll
  for (int q = 0; q < W::KTW; ++q)
#pragma unroll
    for (int vb = 0; vb < W::VBW; ++vb) {
      const int k = 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g;
      out4<F32>(ro, (16 * (W::vb0(w) + vb) + n) * f.dk + k, f.dk - k, a.vec_k != 0, acc[q][vb]);
    }
}

// slot ch := decay^{L_ch} (state before) + slot ch: the state after every chunk, one
// thread per state element, eight loads ahead; also memory_out and snapshots.
template <class E>
__global__ __launch_bounds__(PNT) void fwd_carry_kernel(const ParArgs a) {
  constexpr int AHEAD = 8;
  const ChunkFwdArgs& f = a.f;
  const int64_t plane = static_cast<int64_t>(f.dv) * f.dk;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * PNT + threadIdx.x;
  if (i >= f.batch * plane) return;
  const int64_t b = i / plane, el = i - b * plane;
  float* slot = a.slots + b * f.n_chunks * plane + el;
  float* snap = f.snapshots != nullptr && f.snapshots != a.slots ? f.snapshots + b * f.n_snap * plane + el : nullptr;
  float x = ld_state<E>(f.memory, i, f.mem_f32 != 0);
  const float decay_c = f.pw[f.chunk], decay_last = f.pw[chunk_tokens(f, f.n_chunks - 1)];
  float buf[AHEAD];
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) buf[j] = j < f.n_chunks ? slot[j * plane] : 0.f;
  int to_snap = f.snap_every, si = 0;
  for (int first = 0; first < f.n_chunks; first += AHEAD) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const int ch = first + j;
      if (ch >= f.n_chunks) break;
      x = fmaf(ch == f.n_chunks - 1 ? decay_last : decay_c, x, buf[j]);
      slot[ch * plane] = x;
      if (snap != nullptr && (--to_snap == 0 || ch == f.n_chunks - 1)) {
        snap[si * plane] = x;
        ++si;
        to_snap = f.snap_every;
      }
      buf[j] = ch + AHEAD < f.n_chunks ? slot[(ch + AHEAD) * plane] : 0.f;
    }
  }
  if (f.memory_out == nullptr) return;
  if (f.mem_f32) static_cast<float*>(f.memory_out)[i] = x;
  else static_cast<typename ET<E>::raw*>(f.memory_out)[i] = ET<E>::from_f(x);
}

template <class E, int DKP>
struct ParShape {
  using raw = typename ET<E>::raw;
  static constexpr int KS = DKP + 4;  // LDS row stride of K, Q (input type) and of M (float32)
  static constexpr int KQ_LOADS = CT * DKP / PNT;
  static constexpr int V_LOADS = CT * PDV / PNT;
  static constexpr int M_LOADS = PDV * DKP / PNT;
  static constexpr size_t kq_bytes = 2ull * CT * KS * sizeof(raw);
  static constexpr size_t v_bytes = 1ull * CT * PVS * sizeof(raw);
  static constexpr size_t m_bytes = 1ull * PDV * KS * 4;
  static constexpr size_t lds_bytes = kq_bytes + v_bytes + m_bytes + PW_N * 4;
  static_assert(lds_bytes <= kMaxLds && kq_bytes % 16 == 0 && v_bytes % 16 == 0, "tiles fit, regions aligned");
};

// The outputs of one chunk, value tiles [split * tiles_per_split, +tiles_per_split).
// Wave w owns tokens [16w, +16).  DIRECT: the starting state (one value tile) is formed
// here and written where a snapshot wants it, and one more workgroup per sequence and
// value tile forms the state after the last chunk.
template <class E, int DKP, bool DIRECT>
__global__ __launch_bounds__(PNT) void fwd_chunk_kernel(const ParArgs a) {
  using S = ParShape<E, DKP>;
  using raw = typename ET<E>::raw;
  constexpr int ES = static_cast<int>(sizeof(raw));
  using W = ParWidth<DKP>;
  constexpr int KS = S::KS, KT = W::KT;
  extern __shared__ __align__(16) unsigned char smem[];
  raw* Ks = reinterpret_cast<raw*>(smem);                            // [CT][KS]
  raw* Qs = Ks + CT * KS;                                            // [CT][KS]
  raw* Vs = reinterpret_cast<raw*>(smem + S::kq_bytes);              // [CT][PVS]
  float* Ms = reinterpret_cast<float*>(smem + S::kq_bytes + S::v_bytes);  // [PDV][KS] starting state
  float* pw = Ms + PDV * KS;

  const ChunkFwdArgs& f = a.f;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.splits));
  const int64_t bc = blockIdx.x / static_cast<unsigned>(a.splits);
  const int per_seq = f.n_chunks + (DIRECT ? 1 : 0);
  const int ch = static_cast<int>(bc % per_seq);
  const int64_t b = bc / per_seq;
  const int dk = f.dk, dv = f.dv;
  const bool past = DIRECT && ch == f.n_chunks;  // the state after the last chunk, no outputs
  const int L = past ? 0 : chunk_tokens(f, ch);
  const int64_t t0 = past ? 0 : b * f.seq_len + static_cast<int64_t>(ch) * f.chunk;
  const bool f32m = f.mem_f32 != 0;
  const int vt_begin = split * a.tiles_per_split;
  const int vt_end = min(vt_begin + a.tiles_per_split, (dv + PDV - 1) / PDV);
  if (tid < PW_N) pw[tid] = f.pw[tid];
  // DIRECT: the first earlier chunk's operands and the initial state, under way with the rest.
  OuterOps<E, DKP> ops;
  f32x4 acc[W::KTW][W::VBW];
  if constexpr (DIRECT) {
    const int v0 = vt_begin * PDV, mb = f32m ? 4 : ES;
    if (ch > 0) ops.load(f, b, 0, v0, w, g, n);
    const __amdgpu_buffer_rsrc_t rm =
        make_rsrc(static_cast<const unsigned char*>(f.memory) + (b * dv + v0) * static_cast<int64_t>(dk) * mb,
                  static_cast<uint32_t>(min(PDV, dv - v0) * dk * mb));
#pragma unroll
    for (int q = 0; q < W::KTW; ++q)
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int k = 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g + r;
          acc[q][vb][r] = ld_mem(rm, (16 * (W::vb0(w) + vb) + n) * dk + k, f32m, k < dk, E());
        }
  }
  {
    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(static_cast<const raw*>(f.keys) + t0 * dk, static_cast<uint32_t>(L * dk * ES));
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(static_cast<const raw*>(f.queries) + t0 * dk, static_cast<uint32_t>(L * dk * ES));
    constexpr int STEP = S::KQ_LOADS < 16 ? S::KQ_LOADS : 16;
#pragma unroll 1
    for (int u0 = 0; u0 < S::KQ_LOADS; u0 += STEP) {
      raw kx[STEP], qx[STEP];
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + PNT * (u0 + u), row = l / DKP, col = l % DKP;
        const int off = col < dk ? (row * dk + col) * ES : kBufOOB;
        kx[u] = buf_load1<E>(rk, off);
        qx[u] = buf_load1<E>(rq, off);
      }
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + PNT * (u0 + u), row = l / DKP, col = l % DKP;
        Ks[row * KS + col] = kx[u];
        Qs[row * KS + col] = qx[u];
      }
    }
  }
  const __amdgpu_buffer_rsrc_t rv =
      make_rsrc(static_cast<const raw*>(f.values) + t0 * dv, static_cast<uint32_t>(L * dv * ES));
  struct Stage {
    raw v[S::V_LOADS];
    float m[DIRECT ? 1 : S::M_LOADS];
  };
  const bool slot_m = !DIRECT && ch > 0;
  const bool m32 = slot_m || f32m;
  const int mb = m32 ? 4 : ES;
  const unsigned char* msrc =
      slot_m ? reinterpret_cast<const unsigned char*>(a.slots + (b * f.n_chunks + ch - 1) * dv * dk)
             : static_cast<const unsigned char*>(f.memory) + b * dv * dk * mb;
  auto load_vtile = [&](int vt, Stage& sg) {
    const int v0 = vt * PDV;
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + PNT * u, row = l / PDV, col = v0 + l % PDV;
      sg.v[u] = buf_load1<E>(rv, col < dv ? (row * dv + col) * ES : kBufOOB);
    }
    if constexpr (!DIRECT) {
      const __amdgpu_buffer_rsrc_t rm =
          make_rsrc(msrc + static_cast<int64_t>(v0) * dk * mb, static_cast<uint32_t>(min(PDV, dv - v0) * dk * mb));
#pragma unroll
      for (int u = 0; u < S::M_LOADS; ++u) {
        const int l = tid + PNT * u, row = l / DKP, col = l % DKP;
        sg.m[u] = ld_mem(rm, row * dk + col, m32, col < dk, E());
      }
    }
  };
  auto store_vtile = [&](const Stage& sg) {
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + PNT * u;
      Vs[(l / PDV) * PVS + l % PDV] = sg.v[u];
    }
    if constexpr (!DIRECT) {
#pragma unroll
      for (int u = 0; u < S::M_LOADS; ++u) {
        const int l = tid + PNT * u;
        Ms[(l / DKP) * KS + l % DKP] = sg.m[u];
      }
    }
  };
  Stage stage;
  load_vtile(vt_begin, stage);
  __syncthreads();  // K, Q, pw

  if constexpr (DIRECT) {
    const int v0 = vt_begin * PDV, rows = min(PDV, dv - v0);
    for (int c = 0; c < ch; ++c) {
      const OuterOps<E, DKP> cur = ops;
      if (c + 1 < ch) ops.load(f, b, c + 1, v0, w, g, n);
      const int Lc = chunk_tokens(f, c);
#pragma unroll
      for (int q = 0; q < W::KTW; ++q)
#pragma unroll
        for (int vb = 0; vb < W::VBW; ++vb) acc[q][vb] *= pw[Lc];
      outer_mac<E, DKP>(cur, Lc, f.c, g, pw, acc);
    }
    // acc is the state after chunk ch - 1
    const bool snap = f.snap_every > 0 && ch > 0 && (past || ch % f.snap_every == 0);
    const bool out = past && f.memory_out != nullptr;
    if (snap || out) {
      const int64_t row0 = static_cast<int64_t>(v0) * dk;
      const int ob = f32m ? 4 : ES;
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc(snap ? f.snapshots + (b * f.n_snap + (ch - 1) / f.snap_every) * dv * dk + row0 : nullptr,
                    snap ? static_cast<uint32_t>(rows * dk * 4) : 0u);
      const __amdgpu_buffer_rsrc_t ro =
          make_rsrc(out ? static_cast<unsigned char*>(f.memory_out) + (b * dv * dk + row0) * ob : nullptr,
                    out ? static_cast<uint32_t>(rows * dk * ob) : 0u);
#pragma unroll
      for (int q = 0; q < W::KTW; ++q)
#pragma unroll
        for (int vb = 0; vb < W::VBW; ++vb) {
          const int k = 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g, el = (16 * (W::vb0(w) + vb) + n) * dk + k;
          out4<F32>(rs, el, dk - k, a.vec_k != 0, acc[q][vb]);
          if (f32m) out4<F32>(ro, el, dk - k, a.vec_k != 0, acc[q][vb]);
          else out4<E>(ro, el, dk - k, a.vec_k != 0, acc[q][vb]);
        }
    }
    if (past) return;
    if (f.hidden != nullptr) {
#pragma unroll
      for (int q = 0; q < W::KTW; ++q)
#pragma unroll
        for (int vb = 0; vb < W::VBW; ++vb)
          *reinterpret_cast<float4*>(Ms + (16 * (W::vb0(w) + vb) + n) * KS + 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g) =
              __builtin_bit_cast(float4, acc[q][vb]);
    }
  }
  if (f.hidden == nullptr) return;

  // S rows of block w: lane (g, n) holds S[i = 16w + n][j = 16 jb + 4 g + r], the operand
  // layout of the product with V below.
  const int irow = 16 * w + n;
  f32x4 qf[KT], p[4];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) p[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < KT; ++kk) {
    qf[kk] = lds_row4<E>(Qs + irow * KS + 16 * kk + 4 * g);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      if (jb <= w) p[jb] = mfma4(lds_row4<E>(Ks + (16 * jb + n) * KS + 16 * kk + 4 * g), qf[kk], p[jb]);
  }
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * jb + 4 * g + r;
      p[jb][r] = j <= irow ? p[jb][r] * (f.c * pw[max(irow - j, 0)]) : 0.f;
    }
  const float sq = pw[irow + 1];
  const __amdgpu_buffer_rsrc_t rh =
      make_rsrc(static_cast<raw*>(f.hidden) + t0 * dv, static_cast<uint32_t>(L * dv * ES));
  for (int vt = vt_begin; vt < vt_end; ++vt) {
    store_vtile(stage);
    if (vt + 1 < vt_end) load_vtile(vt + 1, stage);
    __syncthreads();  // value tile (and state tile) in LDS
#pragma unroll
    for (int vb = 0; vb < 2; ++vb) {
      f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KT; ++kk)
        o = mfma4(lds_row4<F32>(Ms + (16 * vb + n) * KS + 16 * kk + 4 * g), qf[kk], o);
      o *= sq;
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= w) o = mfma4(lds_col4<E>(Vs + (16 * jb + 4 * g) * PVS + 16 * vb + n, PVS), p[jb], o);
      const int v = vt * PDV + 16 * vb + 4 * g;
      out4<E>(rh, irow * dv + v, dv - v, a.vec_v != 0, o);
    }
    if (vt + 1 < vt_end) __syncthreads();  // every read of this tile done
  }
}

template <class E, int DKP, bool DIRECT>
int launch_chunks(const ParArgs& a, hipStream_t s) {
  using S = ParShape<E, DKP>;
  if (S::lds_bytes > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_chunk_kernel<E, DKP, DIRECT>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(S::lds_bytes));
    if (e != hipSuccess) {
      set_error("chunk_update_fwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
  }
  hipLaunchKernelGGL((fwd_chunk_kernel<E, DKP, DIRECT>),
                     dim3(static_cast<unsigned>(a.f.batch * (a.f.n_chunks + (DIRECT ? 1 : 0)) * a.splits)), dim3(PNT), S::lds_bytes, s, a);
  return check_launch("chunk_update_fwd(chunks)");
}

template <class E, int DKP>
int launch_par(const ParArgs& a, hipStream_t s) {
  if (a.slots == nullptr) return launch_chunks<E, DKP, true>(a, s);
  const int64_t vtiles = (a.f.dv + PDV - 1) / PDV;
  hipLaunchKernelGGL((fwd_outer_kernel<E, DKP>), dim3(static_cast<unsigned>(a.f.batch * a.f.n_chunks * vtiles)),
                     dim3(PNT), 0, s, a);
  int rc = check_launch("chunk_update_fwd(outer)");
  if (rc != GRM_HIP_OK) return rc;
  const int64_t n = a.f.batch * a.f.dv * static_cast<int64_t>(a.f.dk);
  hipLaunchKernelGGL(fwd_carry_kernel<E>, dim3(static_cast<unsigned>((n + PNT - 1) / PNT)), dim3(PNT), 0, s, a);
  rc = check_launch("chunk_update_fwd(carry)");
  if (rc != GRM_HIP_OK || a.f.hidden == nullptr) return rc;
  return launch_chunks<E, DKP, false>(a, s);
}

template <class E>
int launch_par_width(const ParArgs& a, hipStream_t s) {
  if (a.f.dk <= 32) return launch_par<E, 32>(a, s);
  if (a.f.dk <= 64) return launch_par<E, 64>(a, s);
  if (a.f.dk <= 128) return launch_par<E, 128>(a, s);
  if constexpr (sizeof(typename ET<E>::raw) == 2) return launch_par<E, 256>(a, s);
  set_error("chunk_update_fwd: key_dim %d exceeds 128 for float32", a.f.dk);
  return GRM_HIP_EUNSUPPORTED;
}

}  // namespace

int64_t par_slot_bytes(int64_t batch, int64_t n_chunks, int64_t value_dim, int64_t key_dim) {
  return batch * n_chunks * value_dim * key_dim * 4;
}

// Up to six chunks, eight of narrow keys, and one workgroup per CU: 4 x 256 tokens (64, 256)
// 15.1 us against 21.1 over slots and 20.6 walked, 4 x 384 (64, 128) 19.1 / 19.3 / 27.4, 4 x 448
// (32, 256) 17.6 / 20.1 / 23.6; eight chunks of 64 keys 26.5 / 22.4 / 35.
bool par_direct(int64_t batch, int64_t n_chunks, int64_t value_dim, int64_t key_dim) {
  return n_chunks <= (key_dim > 32 ? 6 : 8) && batch * (n_chunks + 1) * ((value_dim + PDV - 1) / PDV) <= kParDirectWgs;
}

bool par_fits(int64_t batch, int64_t n_chunks, int64_t value_dim, int64_t key_dim) {
  const int64_t vtiles = (value_dim + PDV - 1) / PDV;
  return batch * (n_chunks + 1) * vtiles <= INT32_MAX && CT * value_dim * 4 <= INT32_MAX &&
         batch * value_dim * key_dim / PNT < INT32_MAX;
}

int launch_scan_par(const ChunkFwdArgs& f, int in_dtype, float* slots, bool vec_k, bool vec_v, hipStream_t s) {
  ParArgs a;
  memset(&a, 0, sizeof(a));
  a.f = f;
  a.slots = slots;
  a.vec_k = vec_k;
  a.vec_v = vec_v;
  const int64_t vtiles = (f.dv + PDV - 1) / PDV, bc = f.batch * f.n_chunks;
  // Direct: one tile per workgroup.  Else two workgroups per CU, as S is repeated by each.
  const int64_t want = slots == nullptr ? vtiles : std::min<int64_t>((512 + bc - 1) / bc, vtiles);
  const int64_t per = (vtiles + want - 1) / want;
  a.tiles_per_split = static_cast<int>(per);
  a.splits = static_cast<int>((vtiles + per - 1) / per);
  switch (in_dtype) {
    case GRM_HIP_F32: return launch_par_width<F32>(a, s);
    case GRM_HIP_F16: return launch_par_width<F16>(a, s);
    default: return launch_par_width<BF16>(a, s);
  }
}

}  // namespace grmhip
