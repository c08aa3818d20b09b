// The chunked scan of a short float32 sequence with its chunks in parallel, gfx950
// (maths and layouts: chunk_scan.hip).
//
// Walking a sequence chunk by chunk costs 3-7 us per 64-token chunk (a chain of LDS
// round trips and float32 MFMAs), on a few workgroups where sequences and value tiles are
// few.  Here a workgroup takes one chunk: it forms the state at the chunk's start itself,
// by walking the earlier chunks' K and V (no S, no outputs), then its outputs; one more per
// sequence forms the last state.  One launch, no workspace.  Bound by the loads' latency.
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

struct ParArgs {
  ChunkFwdArgs f;
  int v_tiles;       // 32-column value tiles
  int vec_k, vec_v;  // rows allow 4-element stores
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
template <int DKP>
struct OuterOps {
  using W = ParWidth<DKP>;
  float k[W::KTW][4][4], v[W::VBW][4][4];
  __device__ __forceinline__ void load(const ChunkFwdArgs& f, int64_t b, int ch, int v0, int w, int g, int n) {
    const int dk = f.dk, dv = f.dv, L = chunk_tokens(f, ch);
    const int64_t t0 = b * f.seq_len + static_cast<int64_t>(ch) * f.chunk;
    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(static_cast<const float*>(f.keys) + t0 * dk, static_cast<uint32_t>(L * dk * 4));
    const __amdgpu_buffer_rsrc_t rv =
        make_rsrc(static_cast<const float*>(f.values) + t0 * dv, static_cast<uint32_t>(L * dv * 4));
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int j = 16 * ib + 4 * g + s;
#pragma unroll
        for (int q = 0; q < W::KTW; ++q) {
          const int kc = 16 * (W::kt0(w) + W::KSTEP * q) + n;
          k[q][ib][s] = buf_load1<F32>(rk, kc < dk ? (j * dk + kc) * 4 : kBufOOB);
        }
#pragma unroll
        for (int vb = 0; vb < W::VBW; ++vb) {
          const int vc = v0 + 16 * (W::vb0(w) + vb) + n;
          v[vb][ib][s] = buf_load1<F32>(rv, vc < dv ? (j * dv + vc) * 4 : kBufOOB);
        }
      }
  }
};

// acc[q][vb] += K^T (w V), w_j = c decay^{L-1-j}; lane (g, n) of a result holds keys
// 16 kt + 4 g + r of value 16 vb + n.
template <int DKP>
__device__ __forceinline__ void outer_mac(const OuterOps<DKP>& x, int L, float c, int g, const float* pw,
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
      for (int vb = 0; vb < W::VBW; ++vb) wv[vb][s] = x.v[vb][ib][s] * wj;
    }
#pragma unroll
    for (int q = 0; q < W::KTW; ++q) {
      f32x4 ka;
#pragma unroll
      for (int s = 0; s < 4; ++s) ka[s] = x.k[q][ib][s];
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb) acc[q][vb] = mfma4(ka, wv[vb], acc[q][vb]);
    }
  }
}

template <int DKP>
struct ParShape {
  static constexpr int KS = DKP + 4;  // LDS row stride of K, Q and M
  static constexpr int KQ_LOADS = CT * DKP / PNT;
  static constexpr int V_LOADS = CT * PDV / PNT;
  static constexpr size_t kq_bytes = 2ull * CT * KS * sizeof(float);
  static constexpr size_t v_bytes = 1ull * CT * PVS * sizeof(float);
  static constexpr size_t m_bytes = 1ull * PDV * KS * 4;
  static constexpr size_t lds_bytes = kq_bytes + v_bytes + m_bytes + PW_N * 4;
  static_assert(lds_bytes <= kMaxLds && kq_bytes % 16 == 0 && v_bytes % 16 == 0, "tiles fit, regions aligned");
};

// One workgroup: the outputs of one chunk for one value tile, from the state at the
// chunk's start, which it forms here and writes where a snapshot wants it; one more
// workgroup per sequence and value tile forms the state after the last chunk.  Wave w owns
// tokens [16w, +16).  Every sum runs in the order of the walk (chunk_fwd_kernel without time
// parts), so float32 results are the walk's, bit for bit.
template <int DKP>
__global__ __launch_bounds__(PNT) void fwd_chunk_kernel(const ParArgs a) {
  using S = ParShape<DKP>;
  using W = ParWidth<DKP>;
  constexpr int KS = S::KS, NKK = DKP / 32;
  extern __shared__ __align__(16) unsigned char smem[];
  float* Ks = reinterpret_cast<float*>(smem);                             // [CT][KS]
  float* Qs = Ks + CT * KS;                                               // [CT][KS]
  float* Vs = reinterpret_cast<float*>(smem + S::kq_bytes);               // [CT][PVS]
  float* Ms = reinterpret_cast<float*>(smem + S::kq_bytes + S::v_bytes);  // [PDV][KS] starting state
  float* pw = Ms + PDV * KS;

  const ChunkFwdArgs& f = a.f;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int v0 = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.v_tiles)) * PDV;
  const int64_t bc = blockIdx.x / static_cast<unsigned>(a.v_tiles);
  const int per_seq = f.n_chunks + 1;
  const int ch = static_cast<int>(bc % per_seq);
  const int64_t b = bc / per_seq;
  const int dk = f.dk, dv = f.dv;
  const bool past = ch == f.n_chunks;  // the state after the last chunk, no outputs
  const int L = past ? 0 : chunk_tokens(f, ch);
  const int64_t t0 = past ? 0 : b * f.seq_len + static_cast<int64_t>(ch) * f.chunk;
  const int rows = min(PDV, dv - v0);
  if (tid < PW_N) pw[tid] = f.pw[tid];
  // The first earlier chunk's operands and the initial state, under way with the rest.
  OuterOps<DKP> ops;
  if (ch > 0) ops.load(f, b, 0, v0, w, g, n);
  f32x4 acc[W::KTW][W::VBW];
  {
    const __amdgpu_buffer_rsrc_t rm =
        make_rsrc(static_cast<const float*>(f.memory) + (b * dv + v0) * static_cast<int64_t>(dk),
                  static_cast<uint32_t>(rows * dk * 4));
#pragma unroll
    for (int q = 0; q < W::KTW; ++q)
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int k = 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g + r;
          acc[q][vb][r] = buf_load1<F32>(rm, k < dk ? ((16 * (W::vb0(w) + vb) + n) * dk + k) * 4 : kBufOOB);
        }
  }
  {
    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(static_cast<const float*>(f.keys) + t0 * dk, static_cast<uint32_t>(L * dk * 4));
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(static_cast<const float*>(f.queries) + t0 * dk, static_cast<uint32_t>(L * dk * 4));
    const __amdgpu_buffer_rsrc_t rv =
        make_rsrc(static_cast<const float*>(f.values) + t0 * dv, static_cast<uint32_t>(L * dv * 4));
    float vx[S::V_LOADS];
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + PNT * u, row = l / PDV, col = v0 + l % PDV;
      vx[u] = buf_load1<F32>(rv, col < dv ? (row * dv + col) * 4 : kBufOOB);
    }
    constexpr int STEP = S::KQ_LOADS < 16 ? S::KQ_LOADS : 16;
#pragma unroll 1
    for (int u0 = 0; u0 < S::KQ_LOADS; u0 += STEP) {
      float kx[STEP], qx[STEP];
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + PNT * (u0 + u), row = l / DKP, col = l % DKP;
        const int off = col < dk ? (row * dk + col) * 4 : kBufOOB;
        kx[u] = buf_load1<F32>(rk, off);
        qx[u] = buf_load1<F32>(rq, off);
      }
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const int l = tid + PNT * (u0 + u), row = l / DKP, col = l % DKP;
        Ks[row * KS + col] = kx[u];
        Qs[row * KS + col] = qx[u];
      }
    }
#pragma unroll
    for (int u = 0; u < S::V_LOADS; ++u) {
      const int l = tid + PNT * u;
      Vs[(l / PDV) * PVS + l % PDV] = vx[u];
    }
  }
  __syncthreads();  // K, Q, V, pw

  for (int c = 0; c < ch; ++c) {
    const OuterOps<DKP> cur = ops;
    if (c + 1 < ch) ops.load(f, b, c + 1, v0, w, g, n);
    const int Lc = chunk_tokens(f, c);
#pragma unroll
    for (int q = 0; q < W::KTW; ++q)
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb) acc[q][vb] *= pw[Lc];
    outer_mac<DKP>(cur, Lc, f.c, g, pw, acc);
  }
  // acc is the state after chunk ch - 1
  const bool snap = f.snap_every > 0 && ch > 0 && (past || ch % f.snap_every == 0);
  const bool out = past && f.memory_out != nullptr;
  if (snap || out) {
    const int64_t row0 = static_cast<int64_t>(v0) * dk;
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(snap ? f.snapshots + (b * f.n_snap + (ch - 1) / f.snap_every) * dv * dk + row0 : nullptr,
                  snap ? static_cast<uint32_t>(rows * dk * 4) : 0u);
    const __amdgpu_buffer_rsrc_t ro =
        make_rsrc(out ? static_cast<float*>(f.memory_out) + b * dv * dk + row0 : nullptr,
                  out ? static_cast<uint32_t>(rows * dk * 4) : 0u);
#pragma unroll
    for (int q = 0; q < W::KTW; ++q)
#pragma unroll
      for (int vb = 0; vb < W::VBW; ++vb) {
        const int k = 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g, el = (16 * (W::vb0(w) + vb) + n) * dk + k;
        out4<F32>(rs, el, dk - k, a.vec_k != 0, acc[q][vb]);
        out4<F32>(ro, el, dk - k, a.vec_k != 0, acc[q][vb]);
      }
  }
  if (past || f.hidden == nullptr) return;  // uniform over the workgroup
#pragma unroll
  for (int q = 0; q < W::KTW; ++q)
#pragma unroll
    for (int vb = 0; vb < W::VBW; ++vb)
      *reinterpret_cast<float4*>(Ms + (16 * (W::vb0(w) + vb) + n) * KS + 16 * (W::kt0(w) + W::KSTEP * q) + 4 * g) =
          __builtin_bit_cast(float4, acc[q][vb]);

  // S rows of block w: lane (g, n) holds S[i = 16w + n][j = 16 jb + 4 g + r], the operand
  // layout of the product with V below.  A 32-deep step takes keys 32 kk + 8 g + s, s = 0 .. 7.
  const int irow = 16 * w + n;
  f32x4 qf[NKK][2], p[4];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) p[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = 32 * kk + 8 * g + 4 * h;
      qf[kk][h] = lds_row4<F32>(Qs + irow * KS + k);
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= w) p[jb] = mfma4(lds_row4<F32>(Ks + (16 * jb + n) * KS + k), qf[kk][h], p[jb]);
    }
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * jb + 4 * g + r;
      p[jb][r] = j <= irow ? p[jb][r] * (f.c * pw[max(irow - j, 0)]) : 0.f;
    }
  const float sq = irow < L ? pw[irow + 1] : 0.f;
  const __amdgpu_buffer_rsrc_t rh =
      make_rsrc(static_cast<float*>(f.hidden) + t0 * dv, static_cast<uint32_t>(L * dv * 4));
  __syncthreads();  // the starting state
#pragma unroll
  for (int vb = 0; vb < 2; ++vb) {
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o = mfma4(lds_row4<F32>(Ms + (16 * vb + n) * KS + 32 * kk + 8 * g + 4 * h), qf[kk][h], o);
    o *= sq;
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      if (jb <= w) o = mfma4(lds_col4<F32>(Vs + (16 * jb + 4 * g) * PVS + 16 * vb + n, PVS), p[jb], o);
    const int v = v0 + 16 * vb + 4 * g;
    out4<F32>(rh, irow * dv + v, dv - v, a.vec_v != 0, o);
  }
}

template <int DKP>
int launch_chunks(const ParArgs& a, hipStream_t s) {
  using S = ParShape<DKP>;
  if (S::lds_bytes > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_chunk_kernel<DKP>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(S::lds_bytes));
    if (e != hipSuccess) {
      set_error("chunk_update_fwd: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
      return static_cast<int>(e);
    }
  }
  hipLaunchKernelGGL((fwd_chunk_kernel<DKP>),
                     dim3(static_cast<unsigned>(a.f.batch * (a.f.n_chunks + 1) * a.v_tiles)), dim3(PNT), S::lds_bytes,
                     s, a);
  return check_launch("chunk_update_fwd(chunks)");
}

}  // namespace

// Up to six chunks, eight of narrow keys, and one workgroup per CU (each repeats the state
// of all earlier chunks).  Whole call: 4 x 256 tokens (key_dim 64, value_dim 256) 14.5 us
// against 19.8 walked, 4 x 384 (64, 128) 17.9 and 26.5, 4 x 448 (32, 256) 15.8 and 22.4,
// 4 x 192 (128, 128) 17.0 and 26.6, one chunk the same; with 640 workgroups, 32 x 256 (64,
// 128), 29.8 and 22.0.  The host's own time for a call is about 13 us; the kernel's 8 us for
// one chunk and 14 for four of (64, 256).
bool par_direct(int64_t batch, int64_t n_chunks, int64_t value_dim, int64_t key_dim) {
  return n_chunks >= 1 && n_chunks <= (key_dim > 32 ? 6 : 8) && CT * value_dim * 4 <= INT32_MAX &&
         batch * (n_chunks + 1) * ((value_dim + PDV - 1) / PDV) <= 256;
}

int launch_scan_par(const ChunkFwdArgs& f, int in_dtype, bool vec_k, bool vec_v, hipStream_t s) {
  if (in_dtype != GRM_HIP_F32) {
    set_error("chunk_update_fwd: the chunk-parallel scan takes float32 inputs");
    return GRM_HIP_EUNSUPPORTED;
  }
  ParArgs a;
  memset(&a, 0, sizeof(a));
  a.f = f;
  a.v_tiles = (f.dv + PDV - 1) / PDV;
  a.vec_k = vec_k;
  a.vec_v = vec_v;
  if (f.dk <= 32) return launch_chunks<32>(a, s);
  if (f.dk <= 64) return launch_chunks<64>(a, s);
  return launch_chunks<128>(a, s);
}

}  // namespace grmhip
