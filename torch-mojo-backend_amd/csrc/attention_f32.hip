// f32 attention, forward and backward, on v_mfma_f32_16x16x4_f32: head_dim 32,
// 64 or 128, causal or full, one K/V head per query head.  Products, sums,
// probabilities and statistics are f32 throughout.
//
// Bound: the MFMA rate (157 TFLOP/s nominal; a sixteenth of bf16's, so the
// softmax, LDS and HBM traffic hide behind it).  The layout needs no data
// movement between the two products of a step: with S^T = K Q^T, lane group g
// of an accumulator holds keys 4g + e (e = its register) of query lr, and the
// MFMA with k = {4g + e} over the groups takes exactly that register as the B
// operand of O^T = V^T P^T.  The A operand, V^T, comes from the row-major V
// tile: one 16-byte read of 4 consecutive head-dim elements of key 4g + e is
// the operand of 4 fragments (fragment i holds head-dim elements 4r + i).  The
// backward is built the same way from K, V (dQ) and Q, dO (dK, dV).
//
// A block of 4 waves owns 64 queries (or keys), 16 a wave, and walks tiles of
// 32 rows of the other operands, double-buffered in LDS by direct loads whose
// 16-byte chunks are XOR-swizzled by row so that reading one chunk of 16 rows
// and reading 16 chunks of one row both cover all banks once.  16-row waves
// rather than 32: at the sizes of f32 training (4 x 12 heads of 256) they make
// enough blocks, and the operand reads are still a quarter of the LDS rate.
//
// Causal, against the element-per-lane kernels that took these calls:
// [4, 12, 255, 64] forward 105 -> 18.1 us, backward 243 -> 43.2 us; [8, 12, 512,
// 64] 424 -> 70.4 us and 1033 -> 183 us (46 and 44 TFLOP/s, counting the causal
// half).
#include <math.h>

#include "attention_f32.h"
#include "common.h"
#include "mfma.h"

extern __shared__ __attribute__((aligned(16))) char attn_f32_smem[];

namespace mi {
namespace {

constexpr int kNT = 256;   // 4 waves
constexpr int kRow = 32;   // rows per staged tile
constexpr int kBlk = 64;   // queries (or keys) per block
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

template <int D>
struct Tile {
  static constexpr int CH = D / 4;             // 16-byte chunks per row
  static constexpr int BYTES = kRow * D * 4;
  static constexpr int NF = D / 16;            // 16-wide head-dim fragments
  static constexpr int W = D >= 64 ? 4 : 2;    // head-dim elements per transposed read
  static constexpr int H = NF / W;             // transposed reads per row
  static __device__ __forceinline__ int swz(int row) { return D >= 64 ? (row & 15) : ((row >> 1) & 7); }

  // rows row0 .. row0 + 31 (past the end: the last one) of a [rows, D] operand
  static __device__ __forceinline__ void load(const float* src, int64_t stride, int64_t row0, int64_t rows, char* dst) {
    constexpr int RPI = 64 / CH;  // rows per wave instruction
    const int lane = threadIdx.x & 63, wave = wave_id();
    const unsigned lds = lds_base_of(dst) + wave * 1024;
#pragma unroll
    for (int it = 0; it < D / 32; ++it) {
      const int r = (it * 4 + wave) * RPI + lane / CH;
      dma_b128(src + min(row0 + r, rows - 1) * stride + ((lane % CH) ^ swz(r)) * 4, lds + it * 4096);
    }
  }
  // lane (lr, lg): 4 consecutive elements 16 ks + 4 lg of row r
  static __device__ __forceinline__ f32x4 row(const char* t, int r, int ks, int lg) {
    return *(const f32x4*)(t + r * (D * 4) + (((ks * 4 + lg) ^ swz(r)) << 4));
  }
  // lane lr: the elements W lr + i of row r in fragments h W + i
  static __device__ __forceinline__ void cols(const char* t, int r, int lr, float (&f)[NF]) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      if constexpr (W == 4) {
        const f32x4 v = *(const f32x4*)(t + r * (D * 4) + (((h * 16 + lr) ^ swz(r)) << 4));
#pragma unroll
        for (int i = 0; i < 4; ++i) f[h * 4 + i] = v[i];
      } else {
        const float2 v = *(const float2*)(t + r * (D * 4) + (((lr >> 1) ^ swz(r)) << 4) + (lr & 1) * 8);
        f[0] = v.x, f[1] = v.y;
      }
    }
  }
  // Write a wave's [D, 16] accumulators (column lr) times `f` to the row at p.
  static __device__ __forceinline__ void store(float* p, const f32x4 (&acc)[NF], int lg, float f) {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (W == 4) {
          f32x4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = acc[h * 4 + i][e] * f;
          *(f32x4*)(p + h * 64 + 4 * (4 * lg + e)) = v;
        } else {
          *(float2*)(p + 2 * (4 * lg + e)) = make_float2(acc[0][e] * f, acc[1][e] * f);
        }
      }
  }
};

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Ends a run of MFMAs whose results other instructions read: the compiler
// adds the wait that such a read needs within a basic block, but where a
// branch followed it here it copied a result two instructions after the MFMA
// (the last row of the last fragment came out without its last term).  The
// wait is tied to every result, so nothing can read one before it.
template <int N>
__device__ __forceinline__ void settle(f32x4 (&acc)[N]) {
  asm volatile("s_nop 15" : "+v"(acc[N - 1]));
#pragma unroll
  for (int n = 0; n < N - 1; ++n) asm volatile("" : "+v"(acc[n]));
}

// Block index -> (batch x head, block of the sequence): each XCD (the
// hardware deals blocks to the 8 round robin) takes a contiguous run of heads,
// so a head's tiles are fetched into one L2.
__device__ __forceinline__ void block_of(uint32_t L, uint32_t total, uint32_t per_head, uint32_t* bh, uint32_t* x) {
  const uint32_t xcd = L & 7, q = total >> 3, r = total & 7;
  const uint32_t i = xcd * q + min(xcd, r) + (L >> 3);
  *bh = i / per_head;
  *x = i - *bh * per_head;
}

// s[sub] (16 keys x 16 queries, C layout) = rows of the tile times the
// register fragments q of the wave's 16 columns.  A score is the sum of eight
// partial chains of D / 8 terms (four of 8 at D = 32), added in a tree, as in
// the element-per-lane kernels.  One chain of D terms was further from 64 bits
// than those (2-norm error of O at [4, 4, 64, 128], full: 2.3e-7 there, 3.6e-7
// in one chain, 1.9e-7 in eight; of dQ at [4, 12, 255, 64], causal: 3.4e-7,
// 3.9e-7, 3.2e-7).  The adds take about 5% of the kernels' time ([4, 12, 255,
// 64] forward 17.2 -> 18.1 us, backward 40.7 -> 43.2); four chains 3%, but
// there short sequences stayed up to 2% further off.
template <int D>
constexpr int kChains = D >= 64 ? 8 : 4;
template <int D>
__device__ __forceinline__ void scores(const char* t, const f32x4 (&q)[D / 16], int lr, int lg, f32x4 (&s)[2]) {
  constexpr int N = kChains<D>;
#pragma unroll
  for (int sub = 0; sub < 2; ++sub) {
    f32x4 c[N];
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const f32x4 a = Tile<D>::row(t, sub * 16 + lr, ks, lg);
#pragma unroll
      for (int j = 0; j < 4; ++j) c[(ks * 4 + j) % N] = mma(a[j], q[ks][j], c[(ks * 4 + j) % N]);
    }
#pragma unroll
    for (int w = N / 2; w > 0; w /= 2)
#pragma unroll
      for (int i = 0; i < w; ++i) c[i] += c[i + w];
    s[sub] = c[0];
  }
}

// acc[f] (head-dim fragment f x 16 columns) += tile^T p
template <int D>
__device__ __forceinline__ void accumulate(const char* t, const f32x4 (&p)[2], int lr, int lg,
                                           f32x4 (&acc)[D / 16]) {
#pragma unroll
  for (int sub = 0; sub < 2; ++sub)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float f[D / 16];
      Tile<D>::cols(t, sub * 16 + 4 * lg + e, lr, f);
#pragma unroll
      for (int n = 0; n < D / 16; ++n) acc[n] = mma(f[n], p[sub][e], acc[n]);
    }
  settle(acc);
}

// Sum or maximum over the four lane groups (same lr).
__device__ __forceinline__ float group_sum(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ float group_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}

// This lane's fragments of one row of q, k, v or dO (times f).
template <int D>
__device__ __forceinline__ void load_frags(const float* row, int lg, float f, f32x4 (&x)[D / 16]) {
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) x[ks] = *(const f32x4*)(row + ks * 16 + lg * 4) * f;
}

template <int D>
__global__ void __launch_bounds__(kNT, 2) fwd_f32(AttnF32 p, uint32_t nblk) {
  typedef Tile<D> T;
  char* const lds = attn_f32_smem;  // 2 stages of a K and a V tile
  uint32_t bh, x;
  block_of(blockIdx.x, gridDim.x, nblk, &bh, &x);
  if (p.causal) x = nblk - 1 - x;  // the longest rows first
  const int64_t b = bh / (uint32_t)p.H, h = bh - b * p.H, q0 = (int64_t)x * kBlk;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t w0 = q0 + wave_id() * 16, qi = w0 + lr;
  const float* K = p.k + b * p.k_b + h * p.k_h;
  const float* V = p.v + b * p.v_b + h * p.v_h;
  f32x4 q[T::NF], o[T::NF];
  load_frags<D>(p.q + b * p.q_b + h * p.q_h + min(qi, p.Sq - 1) * p.q_s, lg, p.scale_log2, q);
#pragma unroll
  for (int n = 0; n < T::NF; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const int64_t kend = p.causal ? min(p.Skv, q0 + kBlk) : p.Skv;
  const int64_t wend = p.causal ? min(p.Skv, w0 + 16) : p.Skv;  // keys this wave can see
  T::load(K, p.k_s, 0, p.Skv, lds);
  T::load(V, p.v_s, 0, p.Skv, lds + T::BYTES);
  int cur = 0;
  for (int64_t k0 = 0; k0 < kend; k0 += kRow, cur ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    if (k0 + kRow < kend) {
      T::load(K, p.k_s, k0 + kRow, p.Skv, lds + (cur ^ 1) * 2 * T::BYTES);
      T::load(V, p.v_s, k0 + kRow, p.Skv, lds + (cur ^ 1) * 2 * T::BYTES + T::BYTES);
    }
    if (k0 >= wend) continue;
    const char* kt = lds + cur * 2 * T::BYTES;
    f32x4 s[2];
    scores<D>(kt, q, lr, lg, s);
    if (k0 + kRow > p.Skv || (p.causal && k0 + kRow - 1 > w0)) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t j = k0 + sub * 16 + 4 * lg + e;
          if (j >= p.Skv || (p.causal && j > qi)) s[sub][e] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[sub][e]);
    const float mn = fmaxf(m, group_max(mx));
    const float ref = mn == -INFINITY ? 0.f : mn;  // nothing visible yet
    const float alpha = exp2f(m - ref);
    m = mn;
    float sum = 0.f;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[sub][e] = exp2f(s[sub][e] - ref);
        sum += s[sub][e];
      }
    l = l * alpha + sum;
#pragma unroll
    for (int n = 0; n < T::NF; ++n) o[n] *= alpha;
    accumulate<D>(kt + T::BYTES, s, lr, lg, o);
  }
  l = group_sum(l);
  if (qi >= p.Sq) return;
  T::store(p.o + b * p.o_b + h * p.o_h + qi * p.o_s, o, lg, l > 0.f ? 1.f / l : 0.f);
  if (lg == 0) p.lse[(b * p.H + h) * p.Sq + qi] = l > 0.f ? (m + log2f(l)) * kLn2 : -INFINITY;
}

// D_i = sum_d dO[i, d] O[i, d], in the order of scores(): a lane per partial
// chain, the terms of an MFMA one after another, then the tree.  Where a query
// gives all its weight to one key, O is that key's V and dP - D is zero, as it
// is in exact arithmetic: in another order it is the rounding of both sums
// (one key: dQ and dK 1e-8 of |dO||V| instead of 0; [1, 2, 3, 64] against 135
// keys, causal: 2-norm error of dQ 7.1e-7, 3.8e-7 in the element-per-lane kernels).
template <int D>
__global__ void __launch_bounds__(kNT) delta_f32(AttnF32 p, int64_t rows) {
  constexpr int N = kChains<D>;
  const int64_t row = ((int64_t)blockIdx.x * kNT + threadIdx.x) / N;
  const int c = threadIdx.x % N;
  const bool ok = row < rows;
  float v = 0.f;
  if (ok) {
    const int64_t i = row % p.Sq, bh = row / p.Sq, b = bh / p.H, h = bh % p.H;
    const float* o = p.o + b * p.o_b + h * p.o_h + i * p.o_s;
    const float* d = p.dout + b * p.do_b + h * p.do_h + i * p.do_s;
#pragma unroll
    for (int t = 0; t < D / 4; t += N) {
      const int at = (t + c) / 4 * 16 + (t + c) % 4;
#pragma unroll
      for (int g = 0; g < 16; g += 4) v = fmaf(o[at + g], d[at + g], v);
    }
  }
#pragma unroll
  for (int off = N / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if (ok && c == 0) p.delta[row] = v;
}

// dQ of 64 queries: dS^T = P^T (dP^T - D), dQ^T = scale K^T dS^T.
template <int D>
__device__ __forceinline__ void dq_f32(const AttnF32& p, uint32_t L, uint32_t total, uint32_t nblk) {
  typedef Tile<D> T;
  char* const lds = attn_f32_smem;
  uint32_t bh, x;
  block_of(L, total, nblk, &bh, &x);
  if (p.causal) x = nblk - 1 - x;
  const int64_t b = bh / (uint32_t)p.H, h = bh - b * p.H, q0 = (int64_t)x * kBlk;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t w0 = q0 + wave_id() * 16, qi = w0 + lr, qc = min(qi, p.Sq - 1);
  const float* K = p.k + b * p.k_b + h * p.k_h;
  const float* V = p.v + b * p.v_b + h * p.v_h;
  f32x4 q[T::NF], dO[T::NF], dq[T::NF];
  load_frags<D>(p.q + b * p.q_b + h * p.q_h + qc * p.q_s, lg, p.scale_log2, q);
  load_frags<D>(p.dout + b * p.do_b + h * p.do_h + qc * p.do_s, lg, 1.f, dO);
#pragma unroll
  for (int n = 0; n < T::NF; ++n) dq[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float lse2 = p.lse[(b * p.H + h) * p.Sq + qc] * kLog2e;
  const float di = p.delta[(b * p.H + h) * p.Sq + qc];

  const int64_t kend = p.causal ? min(p.Skv, q0 + kBlk) : p.Skv;
  const int64_t wend = p.causal ? min(p.Skv, w0 + 16) : p.Skv;
  T::load(K, p.k_s, 0, p.Skv, lds);
  T::load(V, p.v_s, 0, p.Skv, lds + T::BYTES);
  int cur = 0;
  for (int64_t k0 = 0; k0 < kend; k0 += kRow, cur ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (k0 + kRow < kend) {
      T::load(K, p.k_s, k0 + kRow, p.Skv, lds + (cur ^ 1) * 2 * T::BYTES);
      T::load(V, p.v_s, k0 + kRow, p.Skv, lds + (cur ^ 1) * 2 * T::BYTES + T::BYTES);
    }
    if (k0 >= wend) continue;
    const char* kt = lds + cur * 2 * T::BYTES;
    f32x4 s[2], dp[2];
    scores<D>(kt, q, lr, lg, s);
    scores<D>(kt + T::BYTES, dO, lr, lg, dp);
    const bool masked = k0 + kRow > p.Skv || (p.causal && k0 + kRow - 1 > w0);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t j = k0 + sub * 16 + 4 * lg + e;
        float pr = exp2f(s[sub][e] - lse2);
        if (masked && (j >= p.Skv || (p.causal && j > qi))) pr = 0.f;
        s[sub][e] = pr * (dp[sub][e] - di);
      }
    accumulate<D>(kt, s, lr, lg, dq);
  }
  if (qi < p.Sq) T::store(p.dq + b * p.dq_b + h * p.dq_h + qi * p.dq_s, dq, lg, p.scale);
}

// dK, dV of 64 keys: dV^T = dO^T P, dK^T = scale Q^T dS.
template <int D>
__device__ __forceinline__ void dkv_f32(const AttnF32& p, uint32_t L, uint32_t total, uint32_t nblk) {
  typedef Tile<D> T;
  char* const lds = attn_f32_smem;                    // 2 stages of a Q and a dO tile
  float* const terms = (float*)(lds + 4 * T::BYTES);  // 2 stages of 32 LSE, 32 D
  uint32_t bh, x;
  block_of(L, total, nblk, &bh, &x);
  const int64_t b = bh / (uint32_t)p.H, h = bh - b * p.H, k0 = (int64_t)x * kBlk;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int64_t w0 = k0 + wave_id() * 16, kj = w0 + lr, kc = min(kj, p.Skv - 1);
  const float* Q = p.q + b * p.q_b + h * p.q_h;
  const float* dO = p.dout + b * p.do_b + h * p.do_h;
  const float* rt = (lane < 32 ? p.lse : p.delta) + (b * p.H + h) * p.Sq;  // this lane's row term
  f32x4 k[T::NF], v[T::NF], dk[T::NF], dv[T::NF];
  load_frags<D>(p.k + b * p.k_b + h * p.k_h + kc * p.k_s, lg, p.scale_log2, k);
  load_frags<D>(p.v + b * p.v_b + h * p.v_h + kc * p.v_s, lg, 1.f, v);
#pragma unroll
  for (int n = 0; n < T::NF; ++n) dk[n] = dv[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int64_t qbeg = p.causal ? k0 : 0;  // a multiple of 32; may lie past the last query
  auto issue = [&](int64_t r0, int st) {
    T::load(Q, p.q_s, r0, p.Sq, lds + st * 2 * T::BYTES);
    T::load(dO, p.do_s, r0, p.Sq, lds + st * 2 * T::BYTES + T::BYTES);
    if (wave_id() == 0) dma_b32(rt + min(r0 + (lane & 31), p.Sq - 1), lds_base_of(terms + st * 64));
  };
  if (qbeg < p.Sq) issue(qbeg, 0);
  int cur = 0;
  for (int64_t r0 = qbeg; r0 < p.Sq; r0 += kRow, cur ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (r0 + kRow < p.Sq) issue(r0 + kRow, cur ^ 1);
    if (p.causal && r0 + kRow - 1 < w0) continue;  // no query of the tile sees this wave's keys
    const char* qt = lds + cur * 2 * T::BYTES;
    f32x4 s[2], dp[2];
    scores<D>(qt, k, lr, lg, s);
    scores<D>(qt + T::BYTES, v, lr, lg, dp);
    const bool masked = r0 + kRow > p.Sq || (p.causal && r0 < w0 + 15);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const f32x4 lse = *(const f32x4*)(terms + cur * 64 + sub * 16 + 4 * lg);
      const f32x4 di = *(const f32x4*)(terms + cur * 64 + 32 + sub * 16 + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t i = r0 + sub * 16 + 4 * lg + e;
        float pr = exp2f(s[sub][e] - lse[e] * kLog2e);
        if (masked && (i >= p.Sq || (p.causal && i < kj))) pr = 0.f;
        s[sub][e] = pr;
        dp[sub][e] = pr * (dp[sub][e] - di[e]);
      }
    }
    accumulate<D>(qt + T::BYTES, s, lr, lg, dv);
    accumulate<D>(qt, dp, lr, lg, dk);
  }
  if (kj >= p.Skv) return;
  T::store(p.dk + b * p.dk_b + h * p.dk_h + kj * p.dk_s, dk, lg, p.scale);
  T::store(p.dv + b * p.dv_b + h * p.dv_h + kj * p.dv_s, dv, lg, 1.f);
}

// Both in one launch: the first `ndkv` blocks do dK and dV, the rest dQ, so
// that one's tail is filled by the other's blocks.
template <int D>
__global__ void __launch_bounds__(kNT, 2) bwd_f32(AttnF32 p, uint32_t ndkv, uint32_t kblk, uint32_t qblk) {
  if (blockIdx.x < ndkv) dkv_f32<D>(p, blockIdx.x, ndkv, kblk);
  else dq_f32<D>(p, blockIdx.x - ndkv, gridDim.x - ndkv, qblk);
}

// Dynamic LDS of a launch; the first launch of a kernel that needs more than
// 64 KB opts it in.
template <int D>
constexpr size_t lds_bytes(bool terms) { return 4 * (size_t)Tile<D>::BYTES + (terms ? 2 * 64 * sizeof(float) : 0); }

bool opt_in(const void* kernel, size_t bytes) {
  return bytes <= 65536 ||
         hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

template <int D>
int run_fwd(const AttnF32& p, hipStream_t s) {
  const uint32_t nblk = ceil_div(p.Sq, kBlk);
  fwd_f32<D><<<(unsigned)(nblk * p.B * p.H), kNT, lds_bytes<D>(false), s>>>(p, nblk);
  return check_launch("mi355x_attn_fwd_gen");
}

template <int D>
int run_bwd(const AttnF32& p, hipStream_t s) {
  static const bool ok = opt_in((const void*)bwd_f32<D>, lds_bytes<D>(true));
  if (!ok) return fail(MI355X_ELAUNCH, "mi355x_attn_bwd_gen: cannot reserve %zu bytes of LDS", lds_bytes<D>(true));
  const int64_t rows = p.B * p.H * p.Sq;
  delta_f32<D><<<ceil_div(rows * kChains<D>, kNT), kNT, 0, s>>>(p, rows);
  const uint32_t kblk = ceil_div(p.Skv, kBlk), qblk = ceil_div(p.Sq, kBlk);
  const uint32_t heads = (uint32_t)(p.B * p.H);
  bwd_f32<D><<<(kblk + qblk) * heads, kNT, lds_bytes<D>(true), s>>>(p, kblk * heads, kblk, qblk);
  return check_launch("mi355x_attn_bwd_gen");
}

// Tiles are loaded and rows stored 16 bytes at a time.
bool wide(const void* p, int64_t b, int64_t h, int64_t s) {
  return ((uintptr_t)p & 15) == 0 && b % 4 == 0 && h % 4 == 0 && s % 4 == 0;
}
bool takes(const AttnF32& p) {
  // a launch takes fewer than 2^32 threads in one dimension: bwd_f32's blocks and
  // delta_f32's chains (the general kernels spread heads and batch over the others)
  return p.B * p.H * ((p.Sq + kBlk - 1) / kBlk + (p.Skv + kBlk - 1) / kBlk) < (1ll << 24) &&
         p.B * p.H * p.Sq < (1ll << 29) &&
         wide(p.q, p.q_b, p.q_h, p.q_s) && wide(p.k, p.k_b, p.k_h, p.k_s) && wide(p.v, p.v_b, p.v_h, p.v_s) &&
         wide(p.o, p.o_b, p.o_h, p.o_s);
}

}  // namespace

int attn_f32_fwd(const AttnF32& p, int64_t d, hipStream_t s) {
  if (!takes(p)) return -1;
  if (d == 64) return run_fwd<64>(p, s);
  if (d == 128) return run_fwd<128>(p, s);
  return d == 32 ? run_fwd<32>(p, s) : -1;
}

int attn_f32_bwd(const AttnF32& p, int64_t d, hipStream_t s) {
  if (!takes(p) || !wide(p.dout, p.do_b, p.do_h, p.do_s) || !wide(p.dq, p.dq_b, p.dq_h, p.dq_s) ||
      !wide(p.dk, p.dk_b, p.dk_h, p.dk_s) || !wide(p.dv, p.dv_b, p.dv_h, p.dv_s))
    return -1;
  if (d == 64) return run_bwd<64>(p, s);
  if (d == 128) return run_bwd<128>(p, s);
  return d == 32 ? run_bwd<32>(p, s) : -1;
}

}  // namespace mi
