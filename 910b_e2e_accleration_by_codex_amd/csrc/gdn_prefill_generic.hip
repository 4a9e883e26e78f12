// Chunked gated delta rule for any head dims d_k, d_v in {16, 32, 64, 128} and fp32, bf16 or fp16
// inputs, computed in fp32 throughout (v_mfma_f32_16x16x4_f32): the general form of
// fast_chunk_gated_delta_rule_v2 (src/gdn_chunk_fast2.py:11-62), which takes any float dtype and
// head dims.  The bf16, d = 128 case has its own segment-parallel kernels (gdn_prefill.hip); this
// file has two forms: chunk_generic_kernel, for callers without a workspace, walks each sequence's
// chunks in order, one workgroup per (sequence, value head, slice of 64 value columns), everything of a
// chunk in LDS and the state slice in MFMA accumulators; generic_prep_kernel + generic_chain_kernel
// (below) take the state-independent part out of that walk, through a workspace.
//
// Per 64-token chunk (src/gdn_chunk_fast2.py:31-59):
//   X  = -(beta_i k_i.k_j e^{G_i - G_j})_{i>j},  T = (I - X)^{-1}  (reg_inv64, the chunked prefill's
//        inverse routine),  U = T diag(beta) V,  W = T diag(beta e^G) K,
//   QK = (q_i.k_j e^{G_i - G_j})_{i>=j},  vn = U - W S,  o = diag(e^G) Q S + QK vn,
//   S' = e^{G_last} S + K^T diag(e^{G_last - G}) vn,
// with q scaled by d_k^-1/2 and, with use_qk_l2norm, q and k l2-normalised in their own dtype first
// (src/gdn_chunk_fast.py:17-18: each op rounded to that dtype).  The output is rounded once to the
// input dtype.  A sequence's chunks of fewer than 64 tokens are zero-padded (g = 0, beta = 0), as
// the reference pads T to a multiple of the chunk.
#include "gdn_device.h"
#include "gdn_internal.h"
#include "gdn_inverse.h"

namespace gdn {
namespace gp {
constexpr int CH = 64;   // chunk length
constexpr int NT = 256;  // 4 waves
constexpr int VS = 64;   // value columns per workgroup (16 per wave)
}  // namespace gp

// One element of an input tensor in dtype code `dt` (GDN_F32, GDN_BF16, GDN_F16), and the rounding
// of an fp32 result to that dtype (the result of one torch elementwise op on such a tensor).
__device__ __forceinline__ float ld_any(const void* p, int64_t i, int dt) {
  if (dt == GDN_F32) return reinterpret_cast<const float*>(p)[i];
  if (dt == GDN_BF16) return bf2f(reinterpret_cast<const uint16_t*>(p)[i]);
  return (float)reinterpret_cast<const _Float16*>(p)[i];
}
__device__ __forceinline__ float rnd_any(float x, int dt) {
  if (dt == GDN_F32) return x;
  if (dt == GDN_BF16) return rbf(x);
  return (float)(_Float16)x;
}
__device__ __forceinline__ void st_any(void* p, int64_t i, float x, int dt) {
  if (dt == GDN_F32) reinterpret_cast<float*>(p)[i] = x;
  else if (dt == GDN_BF16) reinterpret_cast<uint16_t*>(p)[i] = f2bf(x);
  else reinterpret_cast<_Float16*>(p)[i] = (_Float16)x;
}

template <int DK>
struct alignas(16) GenSmem {
  static constexpr int LK = DK + 4;  // fp32 row pitches
  static constexpr int LV = gp::VS + 4;
  static constexpr int LC = gp::CH + 4;
  float K[gp::CH * LK];  // key rows (normalised), zero past the chunk's end
  float Q[gp::CH * LK];  // query rows (normalised, times d_k^-1/2)
  float W[gp::CH * LK];  // T diag(beta e^G) K
  float U[gp::CH * LV];  // the slice's value rows, then U = T diag(beta) V
  float T[gp::CH * LC];  // X, then T
  float A[gp::CH * LC];  // QK
  float G[gp::CH], eG[gp::CH], dec[gp::CH], beta[gp::CH];
  float gl;
  float tiles[4 * 16 * kTrPitch];  // wave 0's transpose tiles (reg_inv64)
};

struct GenArgs {
  const void* q;
  const void* k;
  const void* v;
  int64_t qs, ks, vs;  // token strides (elements)
  const float* g;
  const void* beta;
  int beta_dt, in_dt;
  const float* init;
  float* final_state;
  const int32_t* rows;
  int n_rows;
  void* out;  // [tokens, Hv, Dv] in in_dt
  const int32_t* cu;
  int nseq, seq_len, Hqk, Hv, Dv, nslice, use_l2;
};

// Rows 0..63 of a [64, DK] tile: row r = t / 4 by the four lanes t % 4 (DK / 4 columns each, at
// columns 4 m + t % 4).  Reads the chunk's row if it exists (zero otherwise), l2-normalises it in
// the input dtype when asked, scales it by `scale` in fp32 and stores it at dst (pitch ld).
template <int DK>
__device__ __forceinline__ void load_rows_norm(float* dst, int ld, const void* src, int64_t stride, int64_t col0,
                                               int len, int dt, int use_l2, float scale) {
  constexpr int PER = DK / 4;
  const int t = threadIdx.x, r = t >> 2, part = t & 3;
  float x[PER];
#pragma unroll
  for (int m = 0; m < PER; ++m) x[m] = r < len ? ld_any(src, (int64_t)r * stride + col0 + 4 * m + part, dt) : 0.f;
  if (use_l2) {
    float ss = 0.f;
#pragma unroll
    for (int m = 0; m < PER; ++m) ss += rnd_any(x[m] * x[m], dt);
    ss += __shfl_xor(ss, 1, kWave);
    ss += __shfl_xor(ss, 2, kWave);
    const float inv = rnd_any(rsqrt_f(rnd_any(rnd_any(ss, dt) + 1e-6f, dt)), dt);
#pragma unroll
    for (int m = 0; m < PER; ++m) x[m] = rnd_any(x[m] * inv, dt);
  }
#pragma unroll
  for (int m = 0; m < PER; ++m) dst[r * ld + 4 * m + part] = x[m] * scale;
}

// 16x16 block of A B^T over kdim (A rows a0.., B rows b0.., both row-major fp32 in LDS): lane (c, g)
// r = sum_k A[a0 + 4g + r][k] B[b0 + c][k] (the MFMA accumulator layout).
__device__ __forceinline__ f32x4 gram16(const float* A, const float* B, int ld, int kdim, int lane) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int c = lane & 15, g = lane >> 4;
  for (int k0 = 0; k0 < kdim; k0 += 4)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[c * ld + k0 + g], B[c * ld + k0 + g], acc, 0, 0, 0);
  return acc;
}

template <int DK>
__global__ __launch_bounds__(gp::NT) void chunk_generic_kernel(GenArgs P) {
  using namespace gp;
  using Sm = GenSmem<DK>;
  constexpr int LK = Sm::LK, LV = Sm::LV, LC = Sm::LC, NJ = DK / 16;
  __shared__ Sm sm;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63, c = lane & 15, g = lane >> 4;
  const int slice = blockIdx.x % P.nslice, rest = blockIdx.x / P.nslice;
  const int h = rest % P.Hv, s = rest / P.Hv;
  if (s >= P.nseq) return;
  const int hk = h / (P.Hv / P.Hqk);
  const int64_t t_seq = P.cu ? (int64_t)P.cu[s] : (int64_t)s * P.seq_len;
  const int Ls = P.cu ? P.cu[s + 1] - P.cu[s] : P.seq_len;
  const int vc0 = slice * VS;             // first value column of the slice
  const int ncol = P.Dv - vc0 < VS ? P.Dv - vc0 : VS;
  const bool mine = 16 * w < ncol;        // this wave's 16 state columns exist
  const int row = P.init || P.final_state ? state_row(P.rows, P.n_rows, s) : -1;
  const int64_t sbase = ((int64_t)(row < 0 ? 0 : row) * P.Hv + h) * DK * P.Dv;
  // the state slice: S[j] lane (c, g) r = S[16 j + 4 g + r][vc0 + 16 w + c]
  f32x4 S[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      S[j][r] = (P.init && row >= 0 && mine) ? P.init[sbase + (int64_t)(16 * j + 4 * g + r) * P.Dv + vc0 + 16 * w + c]
                                             : 0.f;
  const float qscale = 1.0f / sqrtf((float)DK);
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < Ls; c0 += CH) {
    const int len = Ls - c0 < CH ? Ls - c0 : CH;
    const int64_t tok0 = t_seq + c0;
    // ---- load: K, Q (normalised), the V slice, g and beta; wave 0 also forms the decay
    load_rows_norm<DK>(sm.K, LK, P.k, P.ks, tok0 * P.ks + (int64_t)hk * DK, len, P.in_dt, P.use_l2, 1.f);
    load_rows_norm<DK>(sm.Q, LK, P.q, P.qs, tok0 * P.qs + (int64_t)hk * DK, len, P.in_dt, P.use_l2, qscale);
    for (int i = t; i < CH * VS; i += NT) {
      const int r = i / VS, col = i % VS;
      sm.U[r * LV + col] = (r < len && col < ncol) ? ld_any(P.v, (tok0 + r) * P.vs + (int64_t)h * P.Dv + vc0 + col, P.in_dt)
                                                   : 0.f;
    }
    if (w == 0) {
      const float gv = lane < len ? P.g[(tok0 + lane) * P.Hv + h] : 0.f;
      const float bv = lane < len ? ld_any(P.beta, (tok0 + lane) * P.Hv + h, P.beta_dt) : 0.f;
      const float G = wave_incl_scan(gv);
      const float Gl = __shfl(G, 63, kWave);
      sm.G[lane] = G;
      sm.eG[lane] = expf(G);
      sm.dec[lane] = expf(Gl - G);
      sm.beta[lane] = bv;
      if (lane == 0) sm.gl = expf(Gl);
    }
    __syncthreads();
    // ---- X = -(beta_i k_i.k_j e^{G_i - G_j})_{i>j} into T, QK = (q_i.k_j e^{G_i - G_j})_{i>=j} into A:
    // 16 blocks each (upper blocks written as zero), 8 per wave
    for (int bi = w; bi < 32; bi += 4) {
      const int which = bi >> 4, a = (bi >> 2) & 3, b = bi & 3;  // which: 0 X, 1 QK
      float* M = which ? sm.A : sm.T;
      f32x4 acc = z4;
      if (b <= a) acc = gram16(which ? sm.Q + 16 * a * LK : sm.K + 16 * a * LK, sm.K + 16 * b * LK, LK, DK, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * a + 4 * g + r, j = 16 * b + c;
        const bool in = which ? i >= j : i > j;
        const float d = expf(in ? sm.G[i] - sm.G[j] : 0.f);
        M[i * LC + j] = in ? (which ? acc[r] * d : -sm.beta[i] * acc[r] * d) : 0.f;
      }
    }
    __syncthreads();
    // ---- T = (I - X)^{-1} (wave 0, in registers)
    if (w == 0) {
      f32x4 XT[10], Xd[4], TT[10];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
#pragma unroll
        for (int b = 0; b < a; ++b) XT[tri(a, b)] = *reinterpret_cast<const f32x4*>(&sm.T[(16 * a + c) * LC + 16 * b + 4 * g]);
        XT[tri(a, a)] = z4;
#pragma unroll
        for (int r = 0; r < 4; ++r) Xd[a][r] = sm.T[(16 * a + 4 * g + r) * LC + 16 * a + c];  // zero on and above the diagonal
      }
      reg_inv64(XT, Xd, TT, sm.tiles, lane);
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          *reinterpret_cast<f32x4*>(&sm.T[(16 * a + c) * LC + 16 * b + 4 * g]) = b <= a ? TT[tri(a, b <= a ? b : 0)] : z4;
    }
    __syncthreads();
    // ---- U = T diag(beta) V (token tile w, held until every wave has read V), W = T diag(beta e^G) K
    {
      f32x4 u[VS / 16];
#pragma unroll
      for (int n = 0; n < VS / 16; ++n) u[n] = z4;
      for (int k0 = 0; k0 < 16 * (w + 1); k0 += 4) {  // T is lower: tokens k <= 16 w + 15
        const int kk = k0 + g;
        const float a = sm.T[(16 * w + c) * LC + kk];
        const float bb = sm.beta[kk];
#pragma unroll
        for (int n = 0; n < VS / 16; ++n)
          u[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bb * sm.U[kk * LV + 16 * n + c], u[n], 0, 0, 0);
      }
      for (int n = 0; n < NJ; ++n) {
        f32x4 acc = z4;
        for (int k0 = 0; k0 < 16 * (w + 1); k0 += 4) {
          const int kk = k0 + g;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(sm.T[(16 * w + c) * LC + kk],
                                                     sm.beta[kk] * sm.eG[kk] * sm.K[kk * LK + 16 * n + c], acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.W[(16 * w + 4 * g + r) * LK + 16 * n + c] = acc[r];
      }
      __syncthreads();
#pragma unroll
      for (int n = 0; n < VS / 16; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.U[(16 * w + 4 * g + r) * LV + 16 * n + c] = u[n][r];
    }
    __syncthreads();
    // ---- the chain on this wave's 16 state columns
    if (mine) {
      f32x4 vn[4], o[4];
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        f32x4 p = z4, qs = z4;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          p = rmm(*reinterpret_cast<const f32x4*>(&sm.W[(16 * tb + c) * LK + 16 * j + 4 * g]), S[j], p);
          qs = rmm(*reinterpret_cast<const f32x4*>(&sm.Q[(16 * tb + c) * LK + 16 * j + 4 * g]), S[j], qs);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * tb + 4 * g + r;
          vn[tb][r] = sm.U[i * LV + 16 * w + c] - p[r];
          o[tb][r] = sm.eG[i] * qs[r];
        }
      }
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
#pragma unroll
        for (int tb2 = 0; tb2 <= tb; ++tb2)
          o[tb] = rmm(*reinterpret_cast<const f32x4*>(&sm.A[(16 * tb + c) * LC + 16 * tb2 + 4 * g]), vn[tb2], o[tb]);
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * tb + 4 * g + r;
          if (i < len)
            st_any(P.out, ((tok0 + i) * P.Hv + h) * (int64_t)P.Dv + vc0 + 16 * w + c, o[tb][r], P.in_dt);
        }
      const float gl = sm.gl;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        f32x4 acc = S[j] * gl;
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
          f32x4 kd;  // Dl(Kd_{tb, j}): lane (c, g) r = K[16 tb + 4 g + r][16 j + c] e^{G_last - G}
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * tb + 4 * g + r;
            kd[r] = sm.K[i * LK + 16 * j + c] * sm.dec[i];
          }
          acc = rmm(kd, vn[tb], acc);
        }
        S[j] = acc;
      }
    }
    __syncthreads();
  }
  if (P.final_state && row >= 0 && mine) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        P.final_state[sbase + (int64_t)(16 * j + 4 * g + r) * P.Dv + vc0 + 16 * w + c] = S[j][r];
  }
}


// ============================================================================================
// The same rule in two kernels, through a workspace: everything of a chunk that does not read the
// state in parallel over all (chunk, value head) pairs (generic_prep_kernel), then the state chain
// alone (generic_chain_kernel), one workgroup per (sequence, value head, 16 value columns).
// ============================================================================================
// What bounds it: the chain, serial over the chunks.  chunk_generic_kernel above runs the whole chunk
// inside that chain (31 us a chunk at d = 64, on one workgroup per head); here a chain step is two
// dependent products of 16 token rows against 16 columns (W S, then K^T vn), 1.4 us measured, and the
// rest (K K^T, the inverse, U, W, Q K^T) runs once, on as many workgroups as there are chunks.
// T = 512, H = 4, d = 64, fp32: 247 us -> 25.7 us (12.0 and 14.1 us traced).  Same formulas, fp32 throughout.
//
// The workspace item of a (chunk, value head) holds the chain's operands as MFMA fragments of 64
// lanes x 4 floats (1 KiB, one 16-byte load a lane); lane (c, g) = (l % 16, l / 16), element r:
//   W  [w 4][j DK/16]        W[16 w + c][16 j + 4 g + r]
//   Q  [w 4][j DK/16]        e^{G} q[16 w + c][16 j + 4 g + r]  (q scaled)
//   Kd [i DK/16][tb 4]       e^{G_last - G} K[16 tb + 4 g + r][16 i + c]
//   A  [tri(w, b)]           QK[16 w + c][16 b + 4 g + r], lower blocks
//   U  [n Dv/16][w 4]        U[16 w + 4 g + r][16 n + c]
// then e^{G_last}.
namespace gp {
constexpr int FR = 256;  // floats of a fragment
__host__ __device__ constexpr int64_t item_floats(int dk, int dv) { return 3 * 64 * dk + 10 * FR + 64 * dv + 4; }
// Workspace held at once: the items of a call beyond it are formed in windows of chunks (and groups of
// sequences), the state carried between windows.  256 MiB: what the last-level cache holds, so the
// chain reads its operands from there; a window is then still hundreds of (chunk, head) pairs.
constexpr int64_t kWorkCap = 256ll << 20;
struct Plan {
  int ns, nw, maxch;  // sequences per group, chunks per window, the longest sequence's chunks
  int64_t bytes, carry_at;
};
inline Plan plan(int nseq, int max_len, int Hv, int Dk, int Dv) {
  Plan p;
  p.maxch = (int)(((int64_t)max_len + CH - 1) / CH);
  const int64_t per = (int64_t)Hv * item_floats(Dk, Dv) * 4;
  int64_t ns = kWorkCap / per;
  if (ns > nseq) ns = nseq;
  p.ns = ns < 1 ? 1 : (int)ns;
  int64_t nw = kWorkCap / (per * p.ns);
  if (nw > p.maxch) nw = p.maxch;
  p.nw = nw < 1 ? 1 : (int)nw;
  p.carry_at = (int64_t)p.ns * p.nw * per;
  p.bytes = p.carry_at + (p.nw < p.maxch ? (int64_t)p.ns * Hv * Dk * Dv * 4 : 0);
  return p;
}
}  // namespace gp

struct GenWindow {
  float* work;   // items ((s - s0) nw + ci) Hv + h
  float* carry;  // states between windows [ns, Hv, Dk, Dv], or null with one window
  int s0, ns;    // the group's sequences s0 .. s0 + ns - 1
  int c0, nw;    // the window's chunks c0 .. c0 + nw - 1
  int maxch;     // chunks of the longest sequence as the caller bounds it: no sequence runs past it (the carry
                 // exists for the windows that this bound makes, whatever the device table says)
};

template <int DK>
struct alignas(16) PrepSmem {
  static constexpr int LK = DK + 4;       // 4 (DK + 4) % 64 = 16: column reads of rows 4 g + r hit 64 banks
  static constexpr int LV = gp::VS + 4;
  static constexpr int LC = gp::CH + 4;
  float K[gp::CH * LK];
  float Q[gp::CH * LK];
  float V[gp::CH * LV];
  float T[gp::CH * LC];  // X, then T (lower blocks)
  float G[gp::CH], eG[gp::CH], dec[gp::CH], beta[gp::CH];
  float tiles[4 * 16 * kTrPitch];
};
constexpr int kPrepThreads = 512;

// Four consecutive elements at index i (a multiple of 4 from a head's start); vec: one vector load (the
// tensor's base and token stride keep it aligned), else element by element.
template <int DT>
__device__ __forceinline__ f32x4 ld4_any(const void* p, int64_t i, bool vec) {
  if (vec) {
    if (DT == GDN_F32) return *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + i);
    typedef uint16_t h4 __attribute__((ext_vector_type(4)));
    const h4 x = *reinterpret_cast<const h4*>(reinterpret_cast<const uint16_t*>(p) + i);
    if (DT == GDN_BF16) return f32x4{bf2f(x[0]), bf2f(x[1]), bf2f(x[2]), bf2f(x[3])};
    typedef _Float16 f4 __attribute__((ext_vector_type(4)));
    const f4 y = __builtin_bit_cast(f4, x);
    return f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
  }
  return f32x4{ld_any(p, i, DT), ld_any(p, i + 1, DT), ld_any(p, i + 2, DT), ld_any(p, i + 3, DT)};
}
template <int DT>
__device__ __forceinline__ bool vec4_ok(const void* p, int64_t stride) {
  return stride % 4 == 0 && reinterpret_cast<uintptr_t>(p) % (DT == GDN_F32 ? 16 : 8) == 0;
}
// A [64, COLS] tile over 512 threads, 4 columns a lane: COLS / 4 lanes a row, PASS rows a thread.
template <int COLS>
struct RowTile {
  static constexpr int LR = COLS / 4, RP = kPrepThreads / LR, PASS = RP >= 64 ? 1 : 64 / RP;
  static __device__ __forceinline__ int row(int p) { return p * RP + (int)threadIdx.x / LR; }  // may be >= 64 (COLS = 16)
  static __device__ __forceinline__ int col() { return 4 * ((int)threadIdx.x % LR); }
};
template <int COLS, int DT>
__device__ __forceinline__ void fetch_tile(f32x4 (&x)[RowTile<COLS>::PASS], const void* src, int64_t stride, int64_t at,
                                           int len, int ncol, bool vec) {
  using R = RowTile<COLS>;
#pragma unroll
  for (int p = 0; p < R::PASS; ++p) {
    const int r = R::row(p);
    x[p] = r < len && R::col() < ncol ? ld4_any<DT>(src, at + (int64_t)r * stride + R::col(), vec) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}
// Rows l2-normalised in the input dtype when asked (as load_rows_norm), times `scale`, into dst.
template <int COLS, int DT>
__device__ __forceinline__ void store_tile_norm(float* dst, int ld, f32x4 (&x)[RowTile<COLS>::PASS], int use_l2,
                                                float scale) {
  using R = RowTile<COLS>;
#pragma unroll
  for (int p = 0; p < R::PASS; ++p) {
    if (use_l2) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += rnd_any(x[p][e] * x[p][e], DT);
#pragma unroll
      for (int o = 1; o < R::LR; o <<= 1) ss += __shfl_xor(ss, o, kWave);
      const float inv = rnd_any(rsqrt_f(rnd_any(rnd_any(ss, DT) + 1e-6f, DT)), DT);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[p][e] = rnd_any(x[p][e] * inv, DT);
    }
    if (R::row(p) < 64) *reinterpret_cast<f32x4*>(&dst[R::row(p) * ld + R::col()]) = x[p] * scale;
  }
}

// One workgroup (8 waves) per (chunk of the window, sequence, value head).  Latency-bound (one wave's
// dependent MFMAs and LDS trips per phase), so the blocks of a phase are dealt over 8 waves and every
// input's loads go out before the first is used; with 4 waves and 4-byte loads it took 15.3 us on 32
// workgroups (T = 512, H = 4, d = 64), with 8 and 16-byte loads 12.0 us.  Wave 0 inverts while waves 1-7
// form Q K^T and copy out the q and K fragments; U and W are dealt by column tiles, which balances the
// triangular T.
template <int DK, int DT>
__global__ __launch_bounds__(kPrepThreads) void generic_prep_kernel(GenArgs P, GenWindow W) {
  using namespace gp;
  using Sm = PrepSmem<DK>;
  constexpr int LK = Sm::LK, LV = Sm::LV, LC = Sm::LC, NJ = DK / 16, NW = kPrepThreads / 64;
  __shared__ Sm sm;
  const int t = threadIdx.x, lane = t & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = blockIdx.x % P.Hv, rest = blockIdx.x / P.Hv;
  const int ci = rest % W.nw, s = W.s0 + rest / W.nw;
  const int hk = h / (P.Hv / P.Hqk);
  const int64_t t_seq = P.cu ? (int64_t)P.cu[s] : (int64_t)s * P.seq_len;
  const int Ls = P.cu ? P.cu[s + 1] - P.cu[s] : P.seq_len;
  const int64_t first = (int64_t)(W.c0 + ci) * CH;
  if (first >= Ls) return;
  const int len = Ls - first < CH ? (int)(Ls - first) : CH;
  const int64_t tok0 = t_seq + first;
  float* item = W.work + (((int64_t)(s - W.s0) * W.nw + ci) * P.Hv + h) * item_floats(DK, P.Dv);
  float* fW = item + lane * 4;
  float* fQ = fW + 64 * DK;
  float* fK = fQ + 64 * DK;
  float* fA = fK + 64 * DK;
  float* fU = fA + 10 * FR;
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4 xk[RowTile<DK>::PASS], xq[RowTile<DK>::PASS], xv[RowTile<VS>::PASS];
  float gv = 0.f, bv = 0.f;
  if (w == 0 && lane < len) {
    gv = P.g[(tok0 + lane) * P.Hv + h];
    bv = ld_any(P.beta, (tok0 + lane) * P.Hv + h, P.beta_dt);
  }
  const bool vvec = vec4_ok<DT>(P.v, P.vs);
  auto fetch_v = [&](int vc0) __attribute__((always_inline)) {
    fetch_tile<VS, DT>(xv, P.v, P.vs, tok0 * P.vs + (int64_t)h * P.Dv + vc0, len, P.Dv - vc0, vvec);
  };
  auto store_v = [&]() __attribute__((always_inline)) { store_tile_norm<VS, DT>(sm.V, LV, xv, 0, 1.f); };
  fetch_tile<DK, DT>(xk, P.k, P.ks, tok0 * P.ks + (int64_t)hk * DK, len, DK, vec4_ok<DT>(P.k, P.ks));
  fetch_tile<DK, DT>(xq, P.q, P.qs, tok0 * P.qs + (int64_t)hk * DK, len, DK, vec4_ok<DT>(P.q, P.qs));
  fetch_v(0);
  __builtin_amdgcn_sched_barrier(0);
  if (w == 0) {
    const float G = wave_incl_scan(gv);
    const float Gl = __shfl(G, 63, kWave);
    sm.G[lane] = G;
    sm.eG[lane] = expf(G);
    sm.dec[lane] = expf(Gl - G);
    sm.beta[lane] = bv;
    if (lane == 0) fU[64 * P.Dv] = expf(Gl);
  }
  store_tile_norm<DK, DT>(sm.K, LK, xk, P.use_l2, 1.f);
  store_tile_norm<DK, DT>(sm.Q, LK, xq, P.use_l2, 1.0f / sqrtf((float)DK));
  store_v();
  __syncthreads();
  // rows 16 b .. of K against rows 16 a .. of M: lane (c, g) r = K[16 b + 4 g + r] . M[16 a + c]
  auto gram = [&](const float* M, int a, int b) __attribute__((always_inline)) {
    f32x4 acc = z4;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      acc = rmm(*reinterpret_cast<const f32x4*>(&sm.K[(16 * b + c) * LK + 16 * j + 4 * g]),
                *reinterpret_cast<const f32x4*>(&M[(16 * a + c) * LK + 16 * j + 4 * g]), acc);
    return acc;
  };
  for (int bi = w; bi < 10; bi += NW) {  // X's lower blocks
    const int a = bi < 1 ? 0 : bi < 3 ? 1 : bi < 6 ? 2 : 3, b = bi - tri(a, 0);
    f32x4 x = gram(sm.K, a, b);
    const int i = 16 * a + c;
    const float Gi = sm.G[i], bi_ = sm.beta[i];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * b + 4 * g + r;
      x[r] = i > j ? -bi_ * x[r] * expf(Gi - sm.G[j]) : 0.f;
    }
    *reinterpret_cast<f32x4*>(&sm.T[i * LC + 16 * b + 4 * g]) = x;
  }
  __syncthreads();
  if (w == 0) {
    f32x4 XT[10], Xd[4], TT[10];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int b = 0; b < a; ++b) XT[tri(a, b)] = *reinterpret_cast<const f32x4*>(&sm.T[(16 * a + c) * LC + 16 * b + 4 * g]);
      XT[tri(a, a)] = z4;
#pragma unroll
      for (int r = 0; r < 4; ++r) Xd[a][r] = sm.T[(16 * a + 4 * g + r) * LC + 16 * a + c];
    }
    reg_inv64(XT, Xd, TT, sm.tiles, lane);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b <= a; ++b) *reinterpret_cast<f32x4*>(&sm.T[(16 * a + c) * LC + 16 * b + 4 * g]) = TT[tri(a, b)];
  } else {
    for (int bi = w - 1; bi < 10; bi += NW - 1) {
      const int a = bi < 1 ? 0 : bi < 3 ? 1 : bi < 6 ? 2 : 3, b = bi - tri(a, 0);
      f32x4 x = gram(sm.Q, a, b);
      const int i = 16 * a + c;
      const float Gi = sm.G[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * b + 4 * g + r;
        x[r] = i >= j ? x[r] * expf(Gi - sm.G[j]) : 0.f;
      }
      *reinterpret_cast<f32x4*>(fA + bi * FR) = x;
    }
    for (int f = w - 1; f < 4 * NJ; f += NW - 1) {
      const int a = f / NJ, j = f % NJ;
      *reinterpret_cast<f32x4*>(fQ + f * FR) =
          *reinterpret_cast<const f32x4*>(&sm.Q[(16 * a + c) * LK + 16 * j + 4 * g]) * sm.eG[16 * a + c];
      const int i = f / 4, tb = f % 4;
      f32x4 kd;
#pragma unroll
      for (int r = 0; r < 4; ++r) kd[r] = sm.K[(16 * tb + 4 * g + r) * LK + 16 * i + c] * sm.dec[16 * tb + 4 * g + r];
      *reinterpret_cast<f32x4*>(fK + f * FR) = kd;
    }
  }
  __syncthreads();
  // column tile n of U = T diag(beta) V and of W = T diag(beta e^G) K (W transposed): T is lower, row tile a
  // takes the token blocks kb <= a
  f32x4 bt[4], be[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    bt[kb] = *reinterpret_cast<const f32x4*>(&sm.beta[16 * kb + 4 * g]);
    be[kb] = bt[kb] * *reinterpret_cast<const f32x4*>(&sm.eG[16 * kb + 4 * g]);
  }
  auto t_frag = [&](int a, int kb) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(&sm.T[(16 * a + c) * LC + 16 * kb + 4 * g]);
  };
  for (int vc0 = 0; vc0 < P.Dv; vc0 += VS) {
    const int nt = (P.Dv - vc0 < VS ? P.Dv - vc0 : VS) / 16, nj = vc0 ? 0 : NJ;  // W's tiles go with slice 0's
    if (vc0) {
      __syncthreads();
      store_v();
      __syncthreads();
    }
    if (vc0 + VS < P.Dv) fetch_v(vc0 + VS);
    for (int n = w; n < nt + nj; n += NW) {
      const bool isw = n >= nt;
      const float* src = isw ? sm.K + 16 * (n - nt) + c : sm.V + 16 * n + c;
      const int ld = isw ? LK : LV;
      f32x4 acc[4] = {z4, z4, z4, z4};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const f32x4 sc = isw ? be[kb] : bt[kb];
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = sc[r] * src[(16 * kb + 4 * g + r) * ld];
        if (isw) {
#pragma unroll
          for (int a = kb; a < 4; ++a) acc[a] = rmm(x, t_frag(a, kb), acc[a]);
        } else {
#pragma unroll
          for (int a = kb; a < 4; ++a) acc[a] = rmm(t_frag(a, kb), x, acc[a]);
        }
      }
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<f32x4*>(isw ? fW + (a * NJ + n - nt) * FR : fU + ((vc0 / 16 + n) * 4 + a) * FR) = acc[a];
    }
  }
}

// Waves 0-3 run the chain (token tile w of vn, then state tiles w, w + 4), two LDS barriers a chunk; waves
// 4-7 form the outputs of token tile w - 4 of the chunk before, so that their products fill the matrix
// cores while the chain waits on LDS.  (Outputs of the same chunk, in step with the chain's two phases:
// 16.0 us for 8 chunks at d = 64, against 14.1 us.)  The state (three copies: read by the chain, read by the outputs,
// being written) and vn (two) pass between the waves through LDS, column-major.  A chunk's fragments
// are requested a step ahead.
template <int DK, int DT>
__global__ __launch_bounds__(512) void generic_chain_kernel(GenArgs P, GenWindow W) {
  using namespace gp;
  constexpr int NJ = DK / 16, LS = DK + 4, LT = CH + 4, NI = NJ > 4 ? 2 : 1;
  __shared__ alignas(16) float ST[3][16 * LS];
  __shared__ alignas(16) float VT[2][16 * LT];
  const int t = threadIdx.x, lane = t & 63, c = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), w = wv & 3;
  const int ncol = P.Dv / 16;
  const int n = blockIdx.x % ncol, rest = blockIdx.x / ncol;
  const int h = rest % P.Hv, s = W.s0 + rest / P.Hv;
  const int64_t t_seq = P.cu ? (int64_t)P.cu[s] : (int64_t)s * P.seq_len;
  const int Ls = P.cu ? P.cu[s + 1] - P.cu[s] : P.seq_len;
  const int nch_s = (Ls + CH - 1) / CH, nch = nch_s < W.maxch ? nch_s : W.maxch;
  const int cnt = nch - W.c0 < W.nw ? nch - W.c0 : W.nw;  // chunks of this window
  if (W.c0 > 0 && cnt <= 0) return;                       // the sequence ended in an earlier window
  const int64_t istride = (int64_t)P.Hv * item_floats(DK, P.Dv);
  const float* item0 = W.work + ((int64_t)(s - W.s0) * W.nw * P.Hv + h) * item_floats(DK, P.Dv) + lane * 4;
  if (wv >= 4) {  // ---- outputs
    struct Frags {
      f32x4 q[NJ], a[4];
    };
    auto load = [&](Frags& F, int ci) __attribute__((always_inline)) {
      const float* it = item0 + ci * istride;
#pragma unroll
      for (int j = 0; j < NJ; ++j) F.q[j] = *reinterpret_cast<const f32x4*>(it + 64 * DK + (w * NJ + j) * FR);
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
        if (tb <= w) F.a[tb] = *reinterpret_cast<const f32x4*>(it + 3 * 64 * DK + (w * (w + 1) / 2 + tb) * FR);
    };
    auto outputs = [&](const Frags& F, int ci, bool barriers) __attribute__((always_inline)) {
      const float* sc = ST[ci % 3];
      const float* vc = VT[ci & 1];
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};  // o^T: lane (c, g) r = o[16 w + c][16 n + 4 g + r]
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc = rmm(*reinterpret_cast<const f32x4*>(&sc[c * LS + 16 * j + 4 * g]), F.q[j], acc);
      if (barriers) lds_barrier();
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
        if (tb <= w) acc = rmm(*reinterpret_cast<const f32x4*>(&vc[c * LT + 16 * tb + 4 * g]), F.a[tb], acc);
      const int64_t tok = (int64_t)(W.c0 + ci) * CH + 16 * w + c;
      if (tok < Ls) {
        const int64_t o = ((t_seq + tok) * P.Hv + h) * (int64_t)P.Dv + 16 * n + 4 * g;
        if (DT == GDN_F32) {
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(P.out) + o) = acc;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) st_any(P.out, o + r, acc[r], DT);
        }
      }
      if (barriers) lds_barrier();
    };
    if (cnt <= 0) return;  // (the chain meets no barrier either)
    Frags fa, fb;
    lds_barrier();
    load(fa, 0);
    lds_barrier();
    lds_barrier();
    int ci = 0;  // chunk ci's outputs in the chain's step ci + 1
    for (; ci + 2 < cnt; ci += 2) {
      load(fb, ci + 1);
      outputs(fa, ci, true);
      load(fa, ci + 2);
      outputs(fb, ci + 1, true);
    }
    if (ci + 1 < cnt) {
      load(fb, ci + 1);
      outputs(fa, ci, true);
      outputs(fb, ci + 1, false);
    } else {
      outputs(fa, ci, false);
    }
    return;
  }
  // ---- the chain
  const bool last = nch <= W.c0 + W.nw;
  const int row = P.init || P.final_state ? state_row(P.rows, P.n_rows, s) : -1;
  const int64_t sbase = ((int64_t)(row < 0 ? 0 : row) * P.Hv + h) * DK * P.Dv;
  float* carry = W.carry + ((int64_t)(s - W.s0) * P.Hv + h) * DK * P.Dv;
  const float* src = W.c0 > 0 ? carry : (P.init && row >= 0 ? P.init + sbase : nullptr);
  struct Frags {
    f32x4 w[NJ], k[4 * NI], u;
    float gl;
  };
  auto load = [&](Frags& F, int ci) __attribute__((always_inline)) {
    const float* it = item0 + (ci < cnt ? ci : cnt - 1) * istride;
#pragma unroll
    for (int j = 0; j < NJ; ++j) F.w[j] = *reinterpret_cast<const f32x4*>(it + (w * NJ + j) * FR);
    const float* iu = it + 3 * 64 * DK + 10 * FR;
    F.u = *reinterpret_cast<const f32x4*>(iu + (n * 4 + w) * FR);
    F.gl = iu[64 * P.Dv - lane * 4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (w + 4 * i < NJ)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb)
          F.k[4 * i + tb] = *reinterpret_cast<const f32x4*>(it + 2 * 64 * DK + ((w + 4 * i) * 4 + tb) * FR);
  };
  Frags fa, fb;
  if (cnt > 0) load(fa, 0);
  f32x4 S[NI];  // state tiles w + 4 i: lane (c, g) r = S[16 (w + 4 i) + 4 g + r][16 n + c]
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (w + 4 * i >= NJ) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[i][r] = src ? src[(int64_t)(16 * (w + 4 * i) + 4 * g + r) * P.Dv + 16 * n + c] : 0.f;
    *reinterpret_cast<f32x4*>(&ST[0][c * LS + 16 * (w + 4 * i) + 4 * g]) = S[i];
  }
  auto step = [&](const Frags& F, int ci) __attribute__((always_inline)) {
    const float* sc = ST[ci % 3];
    float* sn = ST[(ci + 1) % 3];
    float* vc = VT[ci & 1];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc = rmm(F.w[j], *reinterpret_cast<const f32x4*>(&sc[c * LS + 16 * j + 4 * g]), acc);
    *reinterpret_cast<f32x4*>(&vc[c * LT + 16 * w + 4 * g]) = F.u - acc;
    lds_barrier();
    f32x4 vn[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) vn[tb] = *reinterpret_cast<const f32x4*>(&vc[c * LT + 16 * tb + 4 * g]);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (w + 4 * i >= NJ) continue;
      S[i] *= F.gl;
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) S[i] = rmm(F.k[4 * i + tb], vn[tb], S[i]);
      *reinterpret_cast<f32x4*>(&sn[c * LS + 16 * (w + 4 * i) + 4 * g]) = S[i];
    }
    lds_barrier();
  };
  if (cnt > 0) {
    __builtin_amdgcn_s_setprio(1);  // over the output wave on the same SIMD
    lds_barrier();
    int ci = 0;
    for (; ci + 1 < cnt; ci += 2) {
      load(fb, ci + 1);
      step(fa, ci);
      load(fa, ci + 2);
      step(fb, ci + 1);
    }
    if (ci < cnt) step(fa, ci);
  }
  float* dst = !last ? carry : (P.final_state && row >= 0 ? P.final_state + sbase : nullptr);
  if (dst) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (w + 4 * i < NJ)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(int64_t)(16 * (w + 4 * i) + 4 * g + r) * P.Dv + 16 * n + c] = S[i][r];
  }
}

template <int DK, int DT>
static void launch_generic_ws(const GenArgs& P, const gp::Plan& pl, float* work, hipStream_t st) {
  float* carry = reinterpret_cast<float*>(reinterpret_cast<char*>(work) + pl.carry_at);
  for (int s0 = 0; s0 < P.nseq; s0 += pl.ns) {
    const int ns = P.nseq - s0 < pl.ns ? P.nseq - s0 : pl.ns;
    int c0 = 0;
    do {  // (no chunks at all: the chain alone hands the initial states on)
      const int nw = pl.maxch - c0 < pl.nw ? pl.maxch - c0 : pl.nw;
      const GenWindow W{work, carry, s0, ns, c0, nw < 1 ? 1 : nw, pl.maxch};
      if (nw > 0) generic_prep_kernel<DK, DT><<<(unsigned)((int64_t)ns * nw * P.Hv), kPrepThreads, 0, st>>>(P, W);
      generic_chain_kernel<DK, DT><<<(unsigned)((int64_t)ns * P.Hv * (P.Dv / 16)), 512, 0, st>>>(P, W);
      c0 += pl.nw;
    } while (c0 < pl.maxch);
  }
}
template <int DK>
static void launch_generic_dt(const GenArgs& P, const gp::Plan& pl, float* work, hipStream_t st) {
  if (P.in_dt == GDN_F32) launch_generic_ws<DK, GDN_F32>(P, pl, work, st);
  else if (P.in_dt == GDN_BF16) launch_generic_ws<DK, GDN_BF16>(P, pl, work, st);
  else launch_generic_ws<DK, GDN_F16>(P, pl, work, st);
}

}  // namespace gdn

using namespace gdn;

namespace {
// The argument checks of both generic entry points (`name` in the messages).
int check_generic(const char* name, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                  int64_t v_stride, const float* g, const void* beta, int beta_dtype, const int32_t* state_rows,
                  int n_rows, const void* out, int64_t total_tokens, const int32_t* cu_seqlens, int nseq, int seq_len,
                  int Hqk, int Hv, int Dk, int Dv, int in_dtype) {
  GDN_REQUIRE(q && k && v && g && beta && out, "%s: null input/output pointer", name);
  GDN_SUPPORT(Dk == 16 || Dk == 32 || Dk == 64 || Dk == 128, "%s: d_k %d unsupported (16, 32, 64 or 128)", name, Dk);
  GDN_SUPPORT(Dv == 16 || Dv == 32 || Dv == 64 || Dv == 128, "%s: d_v %d unsupported (16, 32, 64 or 128)", name, Dv);
  GDN_REQUIRE(in_dtype == GDN_F32 || in_dtype == GDN_BF16 || in_dtype == GDN_F16, "%s: bad q/k/v dtype", name);
  GDN_REQUIRE(beta_dtype == GDN_F32 || beta_dtype == GDN_BF16 || beta_dtype == GDN_F16, "%s: bad beta dtype", name);
  GDN_REQUIRE(Hqk > 0 && Hv > 0 && Hv % Hqk == 0, "%s: bad heads Hqk=%d Hv=%d", name, Hqk, Hv);
  GDN_REQUIRE(nseq >= 0 && total_tokens >= 0 && seq_len >= 0, "%s: negative sizes", name);
  GDN_REQUIRE(cu_seqlens || (int64_t)nseq * seq_len == total_tokens,
              "%s: without cu_seqlens nseq*seq_len must be total_tokens", name);
  GDN_REQUIRE(state_rows ? n_rows >= 0 : n_rows == nseq, "%s: without state_rows, n_rows must equal nseq", name);
  GDN_REQUIRE(q_stride >= (int64_t)Hqk * Dk && k_stride >= (int64_t)Hqk * Dk && v_stride >= (int64_t)Hv * Dv,
              "%s: token strides too small", name);
  return GDN_OK;
}
}  // namespace

extern "C" int gdn_chunk_prefill_generic(const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                         const void* v, int64_t v_stride, const float* g, const void* beta,
                                         int beta_dtype, const float* initial_state, float* final_state,
                                         const int32_t* state_rows, int n_rows, void* out, int64_t total_tokens,
                                         const int32_t* cu_seqlens, int nseq, int seq_len, int Hqk, int Hv, int Dk,
                                         int Dv, int in_dtype, int use_qk_l2norm, void* stream) {
  clear_error();
  const int rc = check_generic("gdn_chunk_prefill_generic", q, q_stride, k, k_stride, v, v_stride, g, beta, beta_dtype,
                               state_rows, n_rows, out, total_tokens, cu_seqlens, nseq, seq_len, Hqk, Hv, Dk, Dv,
                               in_dtype);
  if (rc) return rc;
  const int nslice = (Dv + gp::VS - 1) / gp::VS;
  const int64_t grid = (int64_t)nseq * Hv * nslice;
  GDN_REQUIRE(grid < (1ll << 31), "gdn_chunk_prefill_generic: grid too large");
  if (nseq == 0) return GDN_OK;
  GenArgs P{q, k, v, q_stride, k_stride, v_stride, g, beta, beta_dtype, in_dtype, initial_state, final_state,
            state_rows, n_rows, out, cu_seqlens, nseq, seq_len, Hqk, Hv, Dv, nslice, use_qk_l2norm};
  hipStream_t st = (hipStream_t)stream;
  switch (Dk) {
    case 16: chunk_generic_kernel<16><<<(unsigned)grid, gp::NT, 0, st>>>(P); break;
    case 32: chunk_generic_kernel<32><<<(unsigned)grid, gp::NT, 0, st>>>(P); break;
    case 64: chunk_generic_kernel<64><<<(unsigned)grid, gp::NT, 0, st>>>(P); break;
    default: chunk_generic_kernel<128><<<(unsigned)grid, gp::NT, 0, st>>>(P); break;
  }
  return check_launch("gdn_chunk_prefill_generic");
}

extern "C" int64_t gdn_chunk_prefill_generic_workspace_bytes(int nseq, int max_len, int Hv, int Dk, int Dv) {
  if (nseq < 0 || max_len < 0 || Hv <= 0 || Dk <= 0 || Dv <= 0) return -1;
  return nseq == 0 ? 0 : gp::plan(nseq, max_len, Hv, Dk, Dv).bytes;
}

extern "C" int gdn_chunk_prefill_generic_ws(const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                            const void* v, int64_t v_stride, const float* g, const void* beta,
                                            int beta_dtype, const float* initial_state, float* final_state,
                                            const int32_t* state_rows, int n_rows, void* out, int64_t total_tokens,
                                            const int32_t* cu_seqlens, int nseq, int seq_len, int Hqk, int Hv, int Dk,
                                            int Dv, int in_dtype, int use_qk_l2norm, void* workspace,
                                            int64_t workspace_bytes, void* stream) {
  clear_error();
  const int rc = check_generic("gdn_chunk_prefill_generic_ws", q, q_stride, k, k_stride, v, v_stride, g, beta,
                               beta_dtype, state_rows, n_rows, out, total_tokens, cu_seqlens, nseq, seq_len, Hqk, Hv,
                               Dk, Dv, in_dtype);
  if (rc) return rc;
  GDN_REQUIRE((int64_t)nseq * seq_len >= total_tokens,
              "gdn_chunk_prefill_generic_ws: seq_len %d cannot bound %d sequences of %lld tokens", seq_len, nseq,
              (long long)total_tokens);
  if (nseq == 0) return GDN_OK;
  const gp::Plan pl = gp::plan(nseq, seq_len, Hv, Dk, Dv);
  GDN_REQUIRE(workspace && aligned(workspace, 16) && workspace_bytes >= pl.bytes,
              "gdn_chunk_prefill_generic_ws: needs a 16-byte aligned workspace of %lld bytes", (long long)pl.bytes);
  GDN_REQUIRE(aligned(out, 16), "gdn_chunk_prefill_generic_ws: out must be 16-byte aligned");
  GDN_REQUIRE((int64_t)pl.ns * pl.nw * Hv < (1ll << 31) && (int64_t)pl.ns * Hv * (Dv / 16) < (1ll << 31),
              "gdn_chunk_prefill_generic_ws: grid too large");
  const GenArgs P{q, k, v, q_stride, k_stride, v_stride, g, beta, beta_dtype, in_dtype, initial_state, final_state,
                  state_rows, n_rows, out, cu_seqlens, nseq, seq_len, Hqk, Hv, Dv, 0, use_qk_l2norm};
  hipStream_t st = (hipStream_t)stream;
  float* work = static_cast<float*>(workspace);
  switch (Dk) {
    case 16: launch_generic_dt<16>(P, pl, work, st); break;
    case 32: launch_generic_dt<32>(P, pl, work, st); break;
    case 64: launch_generic_dt<64>(P, pl, work, st); break;
    default: launch_generic_dt<128>(P, pl, work, st); break;
  }
  return check_launch("gdn_chunk_prefill_generic_ws");
}
