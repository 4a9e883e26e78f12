// GQA decode attention of the hybrid stack's full-attention layers, for N slots of one new token
// each, over a per-slot KV cache: HF Qwen3_5Attention.forward (modeling_qwen3_5.py:629-700) with
// its q/k Qwen3_5RMSNorm, partial rotary (apply_rotary_pos_emb, :554-580), eager attention
// (:604-626) and the sigmoid output gate (:698), as the reference's engine runs it at decode.
//
// HBM-bound on the cache (read once).  Launches:
//   1. attn_prep_kernel, only when the projection comes as split-K partials: one wave per (slot, head
//      row).  RMSNorm (fp32, (1 + w), bf16) of the q and k rows, rotary on the first rd dims (fp32,
//      bf16), q handed on in fp32 (bf16 values: the scores take them as such), k and v written into the cache at
//      the slot's position.
//      With a bf16 projection the split kernel's workgroups do that themselves (each its kv head's q
//      rows, the one holding the slot's position also k and v), under the latency of their cache loads.
//   2. attn_split_kernel: one workgroup per (256-token split, kv head, slot) with the kv head's G query
//      heads.  The whole K block is requested up front and the V block into the registers K leaves (16 KB
//      a wave in flight, 16 waves a CU); the scores, from the transposed K cache [hd, T], and P V, from the
//      V cache [T, hd], run on bf16 MFMA with the G heads as one 16-wide dimension.  Both caches lie
//      across the products' reduction, so a lane transposes the 8 x 4 (K) or 8 x 8 (V) blocks it loaded
//      in registers; the scores come out in the layout P V takes them in, so the softmax needs no
//      exchange but the maximum.
//   3. attn_combine_kernel: per (slot, query head): the splits merged with their max (flash
//      decoding), o rounded to bf16 and multiplied by bf16(sigmoid(gate)).
// Rounding: scores and the softmax's max and exponentials are fp32 (the eager path rounds the scores
// to bf16 too).  The probabilities are rounded to bf16, as the eager path rounds its normalised
// ones, and P V multiplies those bf16 values against bf16 V with fp32 accumulation; the split's
// exp-sum adds the same rounded values.  The test holds the result to an
// fp32 reference.
#include "gdn_device.h"
#include "gdn_internal.h"

namespace gdn {
namespace attn {
// Tokens per split workgroup.  A wave takes 64 tokens by at most 128 dims (its K block, then its V block, is 64
// VGPRs): 4 waves, or 8 at hd = 256.
constexpr int SPLIT = 256;
__host__ __device__ constexpr int split_threads(int hd) { return hd == 256 ? 512 : 256; }
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline int64_t round256(int64_t b) { return (b + 255) / 256 * 256; }
// Two bf16 values a, b (dwords holding two bf16 each) paired as (a.lo, b.lo) / (a.hi, b.hi).
__device__ __forceinline__ uint32_t pair_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t pair_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
__device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// workspace: q (fp32 [N, nh, hd]) | m, l (fp32 [N, nh, S, 2]) | partial o (fp32 [N, nh, S, hd])
struct Work {
  float* q;
  float* ml;
  float* o;
};
__host__ __device__ inline int splits_of(int T) { return (T + SPLIT - 1) / SPLIT; }
__host__ __device__ inline int64_t work_bytes(int N, int nh, int hd, int T) {
  const int64_t S = splits_of(T);
  return round256((int64_t)N * nh * hd * 4) + round256((int64_t)N * nh * S * 2 * 4) +
         round256((int64_t)N * nh * S * hd * 4);
}
__host__ __device__ inline Work work_of(float* base, int N, int nh, int hd, int T) {
  const int64_t S = splits_of(T);
  char* p = reinterpret_cast<char*>(base);
  Work w;
  w.q = reinterpret_cast<float*>(p);
  p += round256((int64_t)N * nh * hd * 4);
  w.ml = reinterpret_cast<float*>(p);
  p += round256((int64_t)N * nh * S * 2 * 4);
  w.o = reinterpret_cast<float*>(p);
  return w;
}
// The fused projection's row n, column col: a bf16 matrix, or bf16(sum of fp32 split-K partials
// [splits][N][width] in split order) -- the same value the reduced projection holds.
struct Src {
  const uint16_t* bf;
  int64_t stride;
  const float* part;
  int splits, N;
  int64_t width;
  __device__ __forceinline__ float operator()(int n, int64_t col) const {
    if (!part) return bf2f(bf[n * stride + col]);
    float s = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < splits; ++sp) s += part[((int64_t)sp * N + n) * width + col];
    return rbf(s);
  }
  // columns col + 64 e, the loads of several splits in flight
  template <int E>
  __device__ __forceinline__ void row(float (&x)[E], int n, int64_t col) const {
    if (!part) {
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = bf2f(bf[n * stride + col + 64 * e]);
      return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = 0.f;
#pragma unroll 4
    for (int sp = 0; sp < splits; ++sp)
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] += part[((int64_t)sp * N + n) * width + col + 64 * e];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = rbf(x[e]);
  }
};
// Lane l's dims l + 64 e of a norm weight (as 1 + w) and, for dims below rd, of the rotary angle's frequency.
template <int HD>
struct NormRope {
  static constexpr int E = HD / 64;
  float w1[E], f[E];
  __device__ __forceinline__ void load(const uint16_t* __restrict__ w, const float* __restrict__ inv_freq, int rd) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int d = lane + 64 * e;
      w1[e] = bf2f(w[d]);
      f[e] = d < rd ? inv_freq[d < rd / 2 ? d : d - rd / 2] : 0.f;
    }
  }
  // f: frequencies -> angles' cosines, sn: their sines, at position p
  __device__ __forceinline__ void angles(float (&sn)[E], int64_t p, int rd) {
    const int lane = threadIdx.x & 63;
    const float fp = (float)p;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      sn[e] = 0.f;
      if (lane + 64 * e < rd) {
        const float ang = fp * f[e];
        sn[e] = sinf(ang);
        f[e] = cosf(ang);
      }
    }
  }
  // x = a head row -> its RMSNorm ((1 + w), rounded to bf16) and rotary (rounded to bf16), one wave; tmp: HD
  // floats of LDS of this wave's own.  The rotary partner of dim d < rd is d +- rd / 2, exchanged through tmp.
  __device__ __forceinline__ void apply(float (&x)[E], const float (&sn)[E], int rd, float eps, float* tmp) const {
    const int lane = threadIdx.x & 63;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) ss += x[e] * x[e];
    ss = wave_sum(ss);
    const float inv = rsqrt_f(ss / (float)HD + eps);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      x[e] = rbf((x[e] * inv) * (1.0f + w1[e]));
      tmp[lane + 64 * e] = x[e];
    }
    // one wave's LDS accesses complete in program order: the partner reads below see the writes
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int half = rd / 2;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int d = lane + 64 * e;
      if (d < rd) {
        const float rot = d < half ? -tmp[d + half] : tmp[d - half];
        x[e] = rbf(x[e] * f[e] + rot * sn[e]);
      }
    }
  }
};
}  // namespace attn

// One wave per (slot n, row r): r < nh are query heads, nh <= r < nh + kv key heads.  Lane l holds
// dims l + 64 e.
template <int HD>
__global__ __launch_bounds__(256) void attn_prep_kernel(attn::Src proj, const int64_t* __restrict__ pos,
                                                        const uint16_t* __restrict__ q_w,
                                                        const uint16_t* __restrict__ k_w,
                                                        const float* __restrict__ inv_freq, uint16_t* __restrict__ kt,
                                                        uint16_t* __restrict__ vc, float* __restrict__ qf, int N,
                                                        int nh, int kv, int rd, int T, float eps) {
  constexpr int E = HD / 64;
  __shared__ float row[4][HD];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + wid;
  if (w >= (int64_t)N * (nh + kv)) return;  // whole waves only: no barrier below
  const int n = (int)(w / (nh + kv)), r = (int)(w % (nh + kv));
  const bool is_q = r < nh;
  const int j = r - nh;
  const int64_t src = is_q ? (int64_t)r * 2 * HD : (int64_t)2 * nh * HD + (int64_t)j * HD;  // row n's column
  const int64_t p = pos[n];
  float x[E], v[E];
  proj.row<E>(x, n, src + lane);
  if (!is_q) proj.row<E>(v, n, (int64_t)2 * nh * HD + (int64_t)kv * HD + (int64_t)j * HD + lane);
  attn::NormRope<HD> nr;
  float sn[E];
  nr.load(is_q ? q_w : k_w, inv_freq, rd);
  nr.angles(sn, p, rd);
  nr.apply(x, sn, rd, eps, row[wid]);
  if (is_q) {
    float* q = qf + ((int64_t)n * nh + r) * HD;
#pragma unroll
    for (int e = 0; e < E; ++e) q[lane + 64 * e] = x[e];
  } else if (p >= 0 && p < T) {
    uint16_t* kd = kt + ((int64_t)n * kv + j) * HD * T + p;
    uint16_t* vd = vc + (((int64_t)n * kv + j) * T + p) * HD;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      kd[(int64_t)(lane + 64 * e) * T] = f2bf(x[e]);
      vd[lane + 64 * e] = f2bf(v[e]);  // exact: the value is bf16
    }
  }
}

// grid (S, kv, N), 4 waves (8 at HD = 256).  Split s covers tokens [SPLIT s, SPLIT s + SPLIT) of the slot's len = pos + 1
// (the new token included).  kPrep: q comes from the bf16 projection (normalised and rotated here), and the
// workgroup that holds position pos forms the new k and v, writes them to the caches and puts them in place of
// what it loaded there; else q is the prep kernel's and the caches hold the new token.
//
// What bounds it: HBM, and how K's rows meet the cache lines (a row of T bf16 values is a whole number of
// lines only where T % 64 == 0).  16 slots of 24 / 4 heads of 256, whole calls (152 MB):
//   contexts 512..4096, T = 4112: 51.6 us with prep and combine kernels around a v_dot2 split kernel of 55 KB of LDS
//   whose V loads waited for the softmax, 38.0 us here; T = 4160: 49.9 -> 36.4 us;
//   contexts 1024: 29.1 -> 23.5 us; 4096: 69.1 -> 54.5 us; 8176: 111.4 -> 88 us (6.1 TB/s).
// On the way: every K and V load up front on v_dot2 (28 VALU instructions per 16 bytes loaded at G = 6, 2 waves a
// SIMD) 68 us; the same on MFMA 59 us; 128-token splits, whose K pieces are half as long, 47 us.
//
// Wave (th, dh) takes tokens 64 th .. + 63 of the split and, at HD = 256, dims 128 dh .. + 127.
//   K: lane (m, g) = (l % 16, l / 16) loads tokens 4 m .. 4 m + 3 of dims 32 s + 8 g + e, e < 8; for each i < 4
//      its 8 values of token 4 m + i are the A fragment (row m) of the product against q (column = head):
//      D_i at lane (head, g), r is the score of token 16 g + 4 r + i.
//   P V: the reduction's slot (g, e) of step u < 2 stands for token 16 g + 8 u + e: lane (head, g) then holds
//      its P operand's 8 values already.  V: lane (m, g) loads dims EV m .. + EV - 1 of tokens 16 g + 8 u + e;
//      for each x < EV its 8 values of dim EV m + x are the B fragment.
template <int HD, int G, bool kPrep>
__global__ __launch_bounds__(attn::split_threads(HD), 4) void attn_split_kernel(attn::Src proj, const int64_t* __restrict__ pos,
                                                         const uint16_t* __restrict__ q_w,
                                                         const uint16_t* __restrict__ k_w,
                                                         const float* __restrict__ inv_freq, uint16_t* kt, uint16_t* vc,
                                                         attn::Work wk, int nh, int kv, int rd, int T,
                                                         float scale, float eps) {
  using namespace attn;
  constexpr int NW = split_threads(HD) / 64;
  constexpr int TH = SPLIT / 64, DH = NW / TH;  // token and dim parts of the waves
  constexpr int DW = HD / DH;                   // dims per wave
  constexpr int KS = DW / 32;                   // 32-dim steps of the scores
  constexpr int EV = DW / 16;                   // dims per lane in P V: 8, or 4 at HD = 64
  constexpr int LQ = HD + 8;                    // row pitch (bf16) of q
  constexpr int E = HD / 64, HPW = (G + NW - 1) / NW;  // q rows per wave
  typedef uint32_t u32v __attribute__((ext_vector_type(EV / 2)));
  __shared__ alignas(16) uint16_t qs[G * LQ];                // q of the G heads
  __shared__ alignas(16) float so[TH][G][HD];                // per token part: P V sums
  __shared__ alignas(16) f32x4 sx[DH == 2 ? NW * 4 * 64 : 1]; // score halves exchanged between the dim parts
  __shared__ float sm[TH][G], sl[TH][G];
  __shared__ float rowt[kPrep ? NW : 1][kPrep ? HD : 1];     // per wave: the rotary exchange
  __shared__ alignas(16) uint16_t knew[kPrep ? HD : 8], vnew[kPrep ? HD : 8];
  const int S = splits_of(T), split = blockIdx.x, j = blockIdx.y, n = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t p = pos[n];
  const int len = (int)(p + 1 < T ? p + 1 : T);
  const int t0 = split * SPLIT;
  if (t0 >= len) return;  // uniform over the workgroup
  const int cnt = len - t0 < SPLIT ? len - t0 : SPLIT;
  const int h0 = j * G, th = wid % TH, d0 = DW * (wid / TH);
  const bool owner = kPrep && p >= t0 && p < t0 + SPLIT && p < T;  // (p >= 0: len > 0)
  const int prel = (int)p - t0 - 64 * th;                          // the position's token in this wave's part
  // ---- the loads q's preparation waits for go out before the cache's (a wave's loads return in order)
  float xq[HPW][E], xk[E], xv[E];
  NormRope<HD> nq, nk;
  if (kPrep) {
#pragma unroll
    for (int i = 0; i < HPW; ++i)
      if (wid + NW * i < G) proj.row<E>(xq[i], n, (int64_t)(h0 + wid + NW * i) * 2 * HD + lane);
    nq.load(q_w, inv_freq, rd);
    if (owner && wid == NW - 1) {
      proj.row<E>(xk, n, (int64_t)2 * nh * HD + (int64_t)j * HD + lane);
      proj.row<E>(xv, n, (int64_t)2 * nh * HD + (int64_t)(kv + j) * HD + lane);
      nk.load(k_w, inv_freq, rd);
    }
  } else {
#pragma unroll
    for (int i = 0; i < HPW; ++i)
      if (wid + NW * i < G)
#pragma unroll
        for (int e = 0; e < E; ++e) xq[i][e] = wk.q[((int64_t)n * nh + h0 + wid + NW * i) * HD + lane + 64 * e];
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- K (tokens past the range: zero).  Cached loads: where T is no multiple of 64 the 128-byte pieces of the
  // waves' 64 tokens straddle cache lines that the next wave reads too (non-temporal: 47.3 us against 42.6 at
  // T = 4112, 2-4% faster where every row is aligned); V's rows are aligned and non-temporal
  u32x2 kr[KS][8];
  {
    const int tl = t0 + 64 * th + 4 * c;
    const uint16_t* kp = kt + (((int64_t)n * kv + j) * HD + d0 + 8 * g4) * T + tl;
    const bool in = tl < ((len + 3) & ~3);  // <= T: T is a multiple of 4
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        kr[s][e] = in ? *reinterpret_cast<const u32x2*>(kp + (int64_t)(32 * s + e) * T) : u32x2{0u, 0u};
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- q into LDS (bf16-exact), and the new token's k and v
  if (kPrep) {
    float sn[E];
    nq.angles(sn, p, rd);
#pragma unroll
    for (int i = 0; i < HPW; ++i)
      if (wid + NW * i < G) nq.apply(xq[i], sn, rd, eps, rowt[wid]);
    if (owner && wid == NW - 1) {
#pragma unroll
      for (int e = 0; e < E; ++e) nk.f[e] = nq.f[e];  // the same angles
      nk.apply(xk, sn, rd, eps, rowt[wid]);
      uint16_t* kd = kt + ((int64_t)n * kv + j) * HD * T + p;
      uint16_t* vd = vc + (((int64_t)n * kv + j) * T + p) * HD;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int d = lane + 64 * e;
        const uint16_t kb = f2bf(xk[e]), vb = f2bf(xv[e]);
        kd[(int64_t)d * T] = kb;
        vd[d] = vb;
        knew[d] = kb;
        vnew[d] = vb;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < HPW; ++i)
    if (wid + NW * i < G)
#pragma unroll
      for (int e = 0; e < E; ++e) qs[(wid + NW * i) * LQ + lane + 64 * e] = f2bf(xq[i][e]);
  lds_barrier();
  if (owner) {  // the cache loads went out before the new token was written: put it in
    const int pt = prel - 4 * c;  // among this lane's K tokens, if in [0, 4)
    if (pt >= 0 && pt < 4) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t b = knew[d0 + 32 * s + 8 * g4 + e];
          const uint32_t x = pt >> 1 ? kr[s][e][1] : kr[s][e][0];
          const uint32_t v = pt & 1 ? (x & 0xffffu) | (b << 16) : (x & 0xffff0000u) | b;
          kr[s][e] = pt >> 1 ? u32x2{kr[s][e][0], v} : u32x2{v, kr[s][e][1]};
        }
    }
  }
  // ---- scores
  const int hq = c < G ? c : G - 1;  // columns past the heads repeat the last (unused)
  f32x4 D[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) D[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const u32x4 q = *reinterpret_cast<const u32x4*>(&qs[hq * LQ + d0 + 32 * s + 8 * g4]);
    u32x4 a[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u32x2 x = kr[s][2 * e], y = kr[s][2 * e + 1];
      a[0][e] = pair_lo(x[0], y[0]);
      a[1][e] = pair_hi(x[0], y[0]);
      a[2][e] = pair_lo(x[1], y[1]);
      a[3][e] = pair_hi(x[1], y[1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) D[i] = mma(a[i], q, D[i]);
  }
  // ---- V, into the registers K leaves.  Rows past the range read as zero (a buffer of the split's rows in range: loads
  // past it return 0): their probability is 0, and 0 times an infinity of a row taken in their place would be NaN
  u32v vr[2][8];
  {
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(vc + (((int64_t)n * kv + j) * T + t0) * HD, 0, cnt * HD * 2, 0x00027000);
    const int at = ((64 * th + 16 * g4) * HD + d0 + EV * c) * 2;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {  // non-temporal
        if constexpr (EV == 8) vr[u][e] = __builtin_amdgcn_raw_buffer_load_b128(rows, at + (8 * u + e) * HD * 2, 0, 2);
        else vr[u][e] = __builtin_amdgcn_raw_buffer_load_b64(rows, at + (8 * u + e) * HD * 2, 0, 2);
      }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (DH == 2) {  // the two dim parts' sums, added in the same order in both
#pragma unroll
    for (int i = 0; i < 4; ++i) sx[(wid * 4 + i) * 64 + lane] = D[i];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i) D[i] = sx[(th * 4 + i) * 64 + lane] + sx[((th + TH) * 4 + i) * 64 + lane];
  }
  // ---- softmax of head c over this wave's 64 tokens
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      D[i][r] = 64 * th + 16 * g4 + 4 * r + i < cnt ? D[i][r] * scale : -INFINITY;
      m = fmaxf(m, D[i][r]);
    }
  m = fmaxf(m, __shfl_xor(m, 16, kWave));
  m = fmaxf(m, __shfl_xor(m, 32, kWave));
  const float m0 = m == -INFINITY ? 0.f : m;  // no token of this part is in range: every probability 0
  float l = 0.f;
  u32x4 pr[2];  // bf16 probabilities: P V's A fragments
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int r = 2 * u + (x >> 1), i = 2 * (x & 1);
      const uint32_t e2 = f2bf2(expf(D[i][r] - m0), expf(D[i + 1][r] - m0));
      pr[u][x] = e2;
      l += __uint_as_float(e2 << 16) + __uint_as_float(e2 & 0xffff0000u);
    }
  l = xor32_sum(xor16_sum(l));
  if (d0 == 0 && lane < G) {
    sm[th][lane] = m;
    sl[th][lane] = l;
  }
  // ---- P V
  if (owner) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (16 * g4 + 8 * u + e == prel) vr[u][e] = *reinterpret_cast<const u32v*>(&vnew[d0 + EV * c]);
  }
  f32x4 O[EV];
#pragma unroll
  for (int x = 0; x < EV; ++x) O[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int x = 0; x < EV / 2; ++x) {
      u32x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = pair_lo(vr[u][2 * e][x], vr[u][2 * e + 1][x]);
        hi[e] = pair_hi(vr[u][2 * e][x], vr[u][2 * e + 1][x]);
      }
      O[2 * x] = mma(pr[u], lo, O[2 * x]);
      O[2 * x + 1] = mma(pr[u], hi, O[2 * x + 1]);
    }
  // O[x] at lane (c, g4), r: head 4 g4 + r, dim d0 + EV c + x
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g4 + r < G) {
#pragma unroll
      for (int x = 0; x < EV; x += 4)
        *reinterpret_cast<f32x4*>(&so[th][4 * g4 + r][d0 + EV * c + x]) = f32x4{O[x][r], O[x + 1][r], O[x + 2][r], O[x + 3][r]};
    }
  lds_barrier();
  // ---- the token parts merged by their maxima
  for (int i = tid; i < G * (HD / 4); i += 64 * NW) {
    const int g = i / (HD / 4), d = 4 * (i % (HD / 4));
    float M = sm[0][g];
#pragma unroll
    for (int x = 1; x < TH; ++x) M = fmaxf(M, sm[x][g]);  // part 0 has the split's first token: finite scores
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
#pragma unroll
    for (int x = 0; x < TH; ++x) {
      const float f = expf(sm[x][g] - M);
      o += *reinterpret_cast<const f32x4*>(&so[x][g][d]) * f;
      L += sl[x][g] * f;
    }
    const int64_t at = ((int64_t)n * nh + h0 + g) * S + split;
    *reinterpret_cast<f32x4*>(&wk.o[at * HD + d]) = o;
    if (d == 0) {
      wk.ml[2 * at] = M;
      wk.ml[2 * at + 1] = L;
    }
  }
}

// grid (N * nh), 256 threads: HD / 4 lanes of 4 dims times GR groups of splits per (slot n, query head h); the
// groups meet in LDS.  4.7 us for 16 x 24 heads of 256, as with one thread per dim walking the splits in turn
// (4.8 us): latency, three loads that wait for one another.  (Partials requested before the maximum is known:
// 5.7 us.)
template <int HD>
__global__ __launch_bounds__(256) void attn_combine_kernel(const int64_t* __restrict__ pos, attn::Src proj,
                                                           attn::Work wk, uint16_t* __restrict__ out,
                                                           int64_t out_stride, int nh, int T) {
  using namespace attn;
  constexpr int LN = HD / 4, GR = 256 / LN;
  __shared__ alignas(16) float so[GR][HD];
  __shared__ float sl[GR];
  const int n = blockIdx.x / nh, h = blockIdx.x % nh, t = threadIdx.x, d4 = t % LN, gr = t / LN;
  const int64_t p = pos[n];
  const int len = (int)(p + 1 < T ? p + 1 : T);
  const int ns = len > 0 ? (len + SPLIT - 1) / SPLIT : 0, S = splits_of(T);
  const float* ml = wk.ml + ((int64_t)n * nh + h) * S * 2;
  const float* op = wk.o + ((int64_t)n * nh + h) * S * HD + 4 * d4;
  const float gate = t < HD ? proj(n, (int64_t)h * 2 * HD + HD + t) : 0.f;
  float M = -INFINITY;
  for (int s = t & 63; s < ns; s += 64) M = fmaxf(M, ml[2 * s]);
  M = wave_max_fast(M);
  float L = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  // the loads of 8 splits at a time are issued together
#pragma unroll 8
  for (int s = gr; s < ns; s += GR) {
    const float f = expf(ml[2 * s] - M);
    L += ml[2 * s + 1] * f;
    o += *reinterpret_cast<const f32x4*>(op + (int64_t)s * HD) * f;
  }
  *reinterpret_cast<f32x4*>(&so[gr][4 * d4]) = o;
  if (d4 == 0) sl[gr] = L;
  __syncthreads();
  if (t >= HD) return;
  float a = 0.f;
  L = 0.f;
#pragma unroll
  for (int x = 0; x < GR; ++x) {
    a += so[x][t];
    L += sl[x];
  }
  a = ns > 0 ? rbf(a / L) : 0.f;  // a negative position attends to nothing: zero output
  out[n * out_stride + (int64_t)h * HD + t] = f2bf(a * bf2f(sigmoid_bf16(gate)));
}

// The arguments of one decode attention call.
struct AttnArgs {
  attn::Src proj;
  const int64_t* pos;
  const uint16_t *q_w, *k_w;
  const float* inv_freq;
  uint16_t *kt, *vc, *out;
  int64_t os;
  int N, nh, kv, rd, T;
  float eps;
};
template <int HD, int G>
static void launch_split(const AttnArgs& A, attn::Work wk, hipStream_t st) {
  const dim3 grid(attn::splits_of(A.T), A.kv, A.N);
  const float scale = 1.0f / sqrtf((float)HD);
  if (A.proj.part)
    attn_split_kernel<HD, G, false><<<grid, attn::split_threads(HD), 0, st>>>(A.proj, A.pos, A.q_w, A.k_w, A.inv_freq, A.kt, A.vc,
                                                                    wk, A.nh, A.kv, A.rd, A.T, scale, A.eps);
  else
    attn_split_kernel<HD, G, true><<<grid, attn::split_threads(HD), 0, st>>>(A.proj, A.pos, A.q_w, A.k_w, A.inv_freq, A.kt, A.vc,
                                                                   wk, A.nh, A.kv, A.rd, A.T, scale, A.eps);
}
template <int HD>
static int launch_all(const AttnArgs& A, float* work, hipStream_t st) {
  const attn::Work wk = attn::work_of(work, A.N, A.nh, HD, A.T);
  const int G = A.nh / A.kv;
  if (G != 1 && G != 2 && G != 4 && G != 6 && G != 8)
    return set_error(GDN_EUNSUP, "gdn_attn_decode: query heads per kv head must be 1, 2, 4, 6 or 8");
  if (A.proj.part) {
    const int64_t waves = (int64_t)A.N * (A.nh + A.kv);
    attn_prep_kernel<HD><<<(unsigned)((waves + 3) / 4), 256, 0, st>>>(A.proj, A.pos, A.q_w, A.k_w, A.inv_freq, A.kt,
                                                                       A.vc, wk.q, A.N, A.nh, A.kv, A.rd, A.T, A.eps);
  }
  switch (G) {
    case 1: launch_split<HD, 1>(A, wk, st); break;
    case 2: launch_split<HD, 2>(A, wk, st); break;
    case 4: launch_split<HD, 4>(A, wk, st); break;
    case 6: launch_split<HD, 6>(A, wk, st); break;
    default: launch_split<HD, 8>(A, wk, st); break;
  }
  attn_combine_kernel<HD><<<A.N * A.nh, 256, 0, st>>>(A.pos, A.proj, wk, A.out, A.os, A.nh, A.T);
  return check_launch("gdn_attn_decode");
}

}  // namespace gdn

using namespace gdn;

extern "C" int64_t gdn_attn_decode_workspace_bytes(int N, int nh, int hd, int T) {
  if (N < 0 || nh < 1 || hd < 1 || T < 1) return -1;
  return attn::work_bytes(N, nh, hd, T);
}

namespace {
int attn_entry(const char* name, attn::Src src, const int64_t* pos, const void* q_norm_w, const void* k_norm_w,
               const float* inv_freq, void* k_cache_t, void* v_cache, void* out, int64_t out_stride, float* work,
               int64_t work_bytes, int N, int nh, int kv, int hd, int rd, int T, float eps, void* stream) {
  GDN_REQUIRE(pos && q_norm_w && k_norm_w && k_cache_t && v_cache && out && work && (inv_freq || rd == 0),
              "%s: null pointer", name);
  GDN_REQUIRE(N >= 0 && nh >= 1 && kv >= 1 && nh % kv == 0, "%s: bad head counts", name);
  GDN_SUPPORT(hd == 64 || hd == 128 || hd == 256, "%s: head_dim must be 64, 128 or 256", name);
  GDN_REQUIRE(rd >= 0 && rd <= hd && rd % 2 == 0, "%s: rotary dims must be even and <= head_dim", name);
  GDN_REQUIRE(T >= 4 && T % 4 == 0, "%s: cache length must be a positive multiple of 4", name);
  GDN_REQUIRE(out_stride >= (int64_t)nh * hd, "%s: output row stride too small", name);
  GDN_REQUIRE(work_bytes >= attn::work_bytes(N, nh, hd, T), "%s: workspace too small (%lld bytes needed)", name,
              (long long)attn::work_bytes(N, nh, hd, T));
  GDN_REQUIRE(aligned(k_cache_t, 8) && aligned(v_cache, 16) && aligned(work, 256) && aligned(pos, 8),
              "%s: K cache 8-byte, V cache 16-byte, workspace 256-byte aligned", name);
  if (N == 0) return GDN_OK;
  src.N = N;
  const AttnArgs A{src, pos, static_cast<const uint16_t*>(q_norm_w), static_cast<const uint16_t*>(k_norm_w), inv_freq,
                   static_cast<uint16_t*>(k_cache_t), static_cast<uint16_t*>(v_cache), static_cast<uint16_t*>(out),
                   out_stride, N, nh, kv, rd, T, eps};
  const hipStream_t st = (hipStream_t)stream;
  switch (hd) {
    case 64: return launch_all<64>(A, work, st);
    case 128: return launch_all<128>(A, work, st);
    default: return launch_all<256>(A, work, st);
  }
}
}  // namespace

extern "C" int gdn_attn_decode(const void* proj, int64_t proj_stride, const int64_t* pos, const void* q_norm_w,
                               const void* k_norm_w, const float* inv_freq, void* k_cache_t, void* v_cache,
                               void* out, int64_t out_stride, float* work, int64_t work_bytes, int N, int nh, int kv,
                               int hd, int rd, int T, float eps, void* stream) {
  clear_error();
  GDN_REQUIRE(proj, "gdn_attn_decode: null pointer");
  GDN_REQUIRE(proj_stride >= (int64_t)(2 * nh + 2 * kv) * hd, "gdn_attn_decode: projection row stride too small");
  const attn::Src src{static_cast<const uint16_t*>(proj), proj_stride, nullptr, 0, N, 0};
  return attn_entry("gdn_attn_decode", src, pos, q_norm_w, k_norm_w, inv_freq, k_cache_t, v_cache, out, out_stride,
                    work, work_bytes, N, nh, kv, hd, rd, T, eps, stream);
}

extern "C" int gdn_attn_decode_partial(const float* part, int splits, const int64_t* pos, const void* q_norm_w,
                                       const void* k_norm_w, const float* inv_freq, void* k_cache_t, void* v_cache,
                                       void* out, int64_t out_stride, float* work, int64_t work_bytes, int N, int nh,
                                       int kv, int hd, int rd, int T, float eps, void* stream) {
  clear_error();
  GDN_REQUIRE(part && splits >= 1 && aligned(part, 4), "gdn_attn_decode_partial: bad partials");
  const attn::Src src{nullptr, 0, part, splits, N, (int64_t)(2 * nh + 2 * kv) * hd};
  return attn_entry("gdn_attn_decode_partial", src, pos, q_norm_w, k_norm_w, inv_freq, k_cache_t, v_cache, out,
                    out_stride, work, work_bytes, N, nh, kv, hd, rd, T, eps, stream);
}
