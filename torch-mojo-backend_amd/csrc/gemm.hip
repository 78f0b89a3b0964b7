// GEMM: C[b] = A[b] * B[b] (+ bias row) (+ C if beta), f32 accumulation.
//
// This file plans a call: which block configuration of the 16-bit MFMA tiles
// (gemm_tile.h), packed copies of operands that cannot be read in place, and
// K splits, whose partials it sums.
//
// Small outputs with a long K (weight gradients) are split along K into f32
// partial tiles in a caller workspace and summed (bias/beta/cast fused) by
// a second pass.  f32 inputs: gemm_f32.hip.
#include <stdio.h>
#include <stdlib.h>

#include "common.h"
#include "gemm.h"
#include "vec.h"

namespace mi {
namespace {

constexpr int kCUs = 256;

// Sum split-K partials: C = sum_s part[s] (+bias) (+C).
__global__ void __launch_bounds__(256) splitk_reduce(GemmArgs g, int splits, int64_t nb) {
  const int64_t mn = g.m * g.n;
  const int64_t total = nb * mn;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int64_t bi = idx / mn, rem = idx % mn;
    const int64_t row = rem / g.n, col = rem % g.n;
    float v = 0.f;
    for (int s = 0; s < splits; ++s) v += g.part[(s * nb + bi) * mn + rem];
    if (g.bias) v += ld_any(g.bias, g.bias_dt, col);
    const int64_t c_es = g.c_dt == MI355X_F32 ? 4 : 2;
    void* Cb = (char*)g.c + bi * g.c_bs * c_es;
    const int64_t off = row * g.c_rs + col;
    if (g.beta) v += ld_any(Cb, g.c_dt, off);
    if (g.round_c) v = round_through(v, g.ab_dt);
    st_any(Cb, g.c_dt, off, v);
  }
}

// splitk_reduce for n % 4 == 0 with 4-aligned C strides and fewer than 2^31
// elements: each thread sums four adjacent columns with 16-byte partial
// loads and 32-bit index math.
template <typename CT>
__device__ __forceinline__ void splitk_reduce4_body(const GemmArgs& g, int splits, int nb, uint32_t blk,
                                                    uint32_t nblk) {
  const uint32_t n4 = (uint32_t)(g.n / 4), mn4 = (uint32_t)g.m * n4;
  const uint32_t total = (uint32_t)nb * mn4;
  const float4* P = (const float4*)g.part;
  for (uint32_t i = blk * 256u + threadIdx.x; i < total; i += nblk * 256u) {
    const uint32_t bi = i / mn4, rem = i - bi * mn4;
    const uint32_t row = rem / n4, col = (rem - row * n4) * 4;
    float4 a = P[i];
    for (int sp = 1; sp < splits; ++sp) {
      const float4 q = P[(uint32_t)sp * total + i];
      a.x += q.x, a.y += q.y, a.z += q.z, a.w += q.w;
    }
    float v[4] = {a.x, a.y, a.z, a.w};
    if (g.bias)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += ld_any(g.bias, g.bias_dt, col + e);
    CT* C = (CT*)g.c + (int64_t)bi * g.c_bs + (int64_t)row * g.c_rs + col;
    float old[4];
    if (g.beta) {
      Vec4<CT>::load(C, old);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += old[e];
    }
    if (g.round_c)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = round_through(v[e], g.ab_dt);
    Vec4<CT>::store(C, v);
  }
}

template <typename CT>
__global__ void __launch_bounds__(256) splitk_reduce4(GemmArgs g, int splits, int nb) {
  splitk_reduce4_body<CT>(g, splits, nb, blockIdx.x, gridDim.x);
}

// Sum the row-sum partials ([slots][nb * m]) into rowsum[batch][m].  A block
// takes 32 rows at a time with 8 threads per row, each summing every 8th
// slot, then combines the 8 in LDS.
__device__ __forceinline__ void rowsum_reduce_body(const GemmArgs& g, int slots, int64_t nb, uint32_t blk,
                                                   uint32_t nblk) {
  __shared__ float red[8][33];
  const int64_t total = nb * g.m;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int64_t base = (int64_t)blk * 32; base < total; base += (int64_t)nblk * 32) {
    const int64_t idx = base + tx;
    float v = 0.f;
    if (idx < total) {
      int s = ty;
      for (; s + 24 < slots; s += 32) {
        const float a0 = g.rs_part[s * total + idx], a1 = g.rs_part[(s + 8) * total + idx];
        const float a2 = g.rs_part[(s + 16) * total + idx], a3 = g.rs_part[(s + 24) * total + idx];
        v += (a0 + a1) + (a2 + a3);
      }
      for (; s < slots; s += 8) v += g.rs_part[s * total + idx];
    }
    red[ty][tx] = v;
    __syncthreads();
    if (ty == 0 && idx < total) {
      float r = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) r += red[j][tx];
      if (g.round_c) r = round_through(r, g.ab_dt);
      st_any(g.rowsum, g.rowsum_dt, idx, r);
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) rowsum_reduce(GemmArgs g, int slots, int64_t nb) {
  rowsum_reduce_body(g, slots, nb, blockIdx.x, gridDim.x);
}

// The two finishing sums of a split-K GEMM with row sums in one launch:
// blocks [0, nbc) sum the C partials, the rest the row-sum partials.
template <typename CT>
__global__ void __launch_bounds__(256) splitk_rowsum_reduce(GemmArgs g, int splits, int nb, int slots,
                                                             uint32_t nbc) {
  if (blockIdx.x < nbc) splitk_reduce4_body<CT>(g, splits, nb, blockIdx.x, nbc);
  else rowsum_reduce_body(g, slots, nb, blockIdx.x - nbc, gridDim.x - nbc);
}

// Pack an operand into a k-contiguous [rows][ld] buffer of 16-bit elements,
// zero-filling k in [K, ld).  Source element (row, k) is at
//   transposed: src + b*sbs + k*sk + row      (row-contiguous source)
//   straight:   src + b*sbs + row*sr + k      (k-contiguous, any row stride)
// 64x64 tiles through LDS keep both the reads and the writes coalesced.
__global__ void __launch_bounds__(256) pack_k_contig(uint16_t* __restrict__ dst, int64_t ld,
                                                     int64_t dst_bs, const uint16_t* __restrict__ src,
                                                     int64_t stride, int64_t sbs, int64_t rows,
                                                     int64_t kdim, int transposed) {
  __shared__ uint16_t tile[64][65];
  const int64_t b = blockIdx.z;
  const int64_t row0 = (int64_t)blockIdx.y * 64, k0 = (int64_t)blockIdx.x * 64;
  const uint16_t* S = src + b * sbs;
  uint16_t* D = dst + b * dst_bs;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (transposed) {
    for (int i = ty; i < 64; i += 4) {  // i: k offset, tx: row offset (contiguous)
      const int64_t k = k0 + i, r = row0 + tx;
      tile[i][tx] = (k < kdim && r < rows) ? S[k * stride + r] : (uint16_t)0;
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {  // i: row offset, tx: k offset (contiguous)
      const int64_t r = row0 + i, k = k0 + tx;
      if (r < rows && k < ld) D[r * ld + k] = tile[tx][i];
    }
  } else {
    for (int i = ty; i < 64; i += 4) {
      const int64_t r = row0 + i, k = k0 + tx;
      if (r < rows && k < ld) D[r * ld + k] = k < kdim ? S[r * stride + k] : (uint16_t)0;
    }
  }
}

// pack_k_contig with 16-byte global accesses, for sources whose base, row or
// k stride and batch stride are 8-element aligned (and, transposed, whose row
// count is a multiple of 8).  A 64x64 tile moves as 512 16-byte chunks, two
// per thread each way.  The LDS tile is [k][row] with a 65-element pitch: the
// 2-byte scatter of a loaded chunk and the 2-byte gather of a stored one then
// hit distinct banks across the wave.
__global__ void __launch_bounds__(256) pack_k_contig_v8(uint16_t* __restrict__ dst, int64_t ld,
                                                        int64_t dst_bs, const uint16_t* __restrict__ src,
                                                        int64_t stride, int64_t sbs, int64_t rows,
                                                        int64_t kdim, int transposed) {
  const int64_t b = blockIdx.z;
  const int64_t row0 = (int64_t)blockIdx.y * 64, k0 = (int64_t)blockIdx.x * 64;
  const uint16_t* S = src + b * sbs;
  uint16_t* D = dst + b * dst_bs;
  const int t = threadIdx.x;
  if (!transposed) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t r = row0 + (t >> 3) + 32 * j, k = k0 + (t & 7) * 8;
      if (r >= rows || k >= ld) continue;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (k + 8 <= kdim) {
        v = *(const uint4*)(S + r * stride + k);
      } else if (k < kdim) {
        uint16_t e8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) e8[e] = k + e < kdim ? S[r * stride + k + e] : (uint16_t)0;
        v = *(const uint4*)e8;
      }
      *(uint4*)(D + r * ld + k) = v;
    }
    return;
  }
  __shared__ uint16_t tile[64][65];  // [k][row]
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int kl = (t >> 3) + 32 * j, rl = (t & 7) * 8;
    const int64_t k = k0 + kl, r = row0 + rl;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (k < kdim && r < rows) v = *(const uint4*)(S + k * stride + r);
    const uint16_t* e8 = (const uint16_t*)&v;
#pragma unroll
    for (int e = 0; e < 8; ++e) tile[kl][rl + e] = e8[e];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int rl = (t >> 3) + 32 * j, kc = (t & 7) * 8;
    const int64_t r = row0 + rl, k = k0 + kc;
    if (r >= rows || k >= ld) continue;
    uint16_t e8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) e8[e] = tile[kc + e][rl];
    *(uint4*)(D + r * ld + k) = *(const uint4*)e8;
  }
}

// ---------------------------------------------------------------------------
// planning
// ---------------------------------------------------------------------------
struct Plan {
  int cfg;  // 0 = C128, 1 = C256, 2 = C192, 3 = C256W, 4 = C64
  int splits;
  int64_t kchunk;
};

// Rows and columns of C per block, and the waves along them.
struct CfgShape {
  int bm, bn, wgn;
};
CfgShape shape_of(int cfg) {
  switch (cfg) {
    case 1: case 3: return {256, 256, 4};
    case 2: return {128, 192, 2};
    case 4: return {64, 64, 2};
    default: return {128, 128, 2};
  }
}

int64_t tiles_of(int cfg, int64_t batch, int64_t m, int64_t n) {
  const CfgShape c = shape_of(cfg);
  return ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * batch;
}

// Row-sum partial slots per split: one per wave column of every column tile.
int64_t rs_slots_of(int cfg, int64_t n) {
  const CfgShape c = shape_of(cfg);
  return (n + c.bn - 1) / c.bn * c.wgn;
}

// Time of `blocks` blocks of a configuration, in units of a full round of C128
// (two blocks on each CU, 0.0141 us per k).  A round that gives a CU one block
// of the two that fit it is shorter (us at K = 768 unless given, C128 / C192 /
// C256 tiles: 4096 x 2304 24.2 / 20.2 / 22.8, 8192 x 2304 40.2 / 32.7 / 46.5,
// 8192 x 3072 45.9 / 40.5 / 48.3, 16384 x 2304 70.7 / 59.7 / 72.2, 16384 x
// 3072 96.4 / 83.7 / 82.0, 2048 x 2304 14.8 / 14.1 / 20.7, 4096 x 768 11.3 /
// 13.9 / 20.7, 16384 x 1024 at K = 1024 38.0 / 49.3 / 33.8).
double rounds_of(int cfg, int64_t blocks) {
  if (cfg == 1) return 1.8 * (double)((blocks + kCUs - 1) / kCUs);
  const double two = cfg == 2 ? 1.45 : 1.0, one = cfg == 2 ? 0.95 : 0.72;
  const int64_t last = blocks % (2 * kCUs);
  return two * (double)(blocks / (2 * kCUs)) + (last == 0 ? 0.0 : last <= kCUs ? one : two);
}

// Time of a plan, in us: its rounds, with K splits the partial sums' way out
// and back and the launch that adds them.
double plan_time(double rounds, int64_t chunk, int64_t splits, int64_t outputs) {
  return rounds * 0.0141 * (double)chunk + (splits > 1 ? 3.0 + (double)(splits + 1) * 4.0 * (double)outputs / 6e6 : 0.0);
}

int64_t chunk_of(int64_t k, int64_t splits) { return ((k + splits - 1) / splits + 63) / 64 * 64; }

// Pick the configuration that finishes in the least time, then split K when
// the output alone cannot fill the chip.
Plan plan_gemm(int64_t batch, int64_t m, int64_t n, int64_t k, bool a_kcontig, bool b_kcontig) {
  Plan best{0, 1, k};
  const int64_t t128 = tiles_of(0, batch, m, n), t256 = tiles_of(1, batch, m, n), t192 = tiles_of(2, batch, m, n);
  double cbest = rounds_of(0, t128);
  // at least three quarters of the CUs busy (2048 x 6912, 216 C256 tiles, K = 1152: 40.4 -> 32.9 us)
  const int64_t fill = kCUs * 3 / 4;
  if (t256 >= (a_kcontig ? fill : kCUs) && rounds_of(1, t256) < cbest) best.cfg = 1, cbest = rounds_of(1, t256);
  if (b_kcontig && t192 >= fill && rounds_of(2, t192) < cbest) best.cfg = 2, cbest = rounds_of(2, t192);
  if (a_kcontig && t128 > kCUs && 2 * t128 < 3 * kCUs && k >= 4096) {
    // A long K under a round that is little more than half full: K splits, if
    // they pay for their partial sums (4096 x 1152 at K = 6912: 97 us; 75 in 3
    // splits of C256, 79 in 2 of C192, 84 in 3 of C128).
    double tbest = 0.9 * cbest * 0.0141 * (double)k;
    for (int cfg = 0; cfg <= (b_kcontig ? 2 : 1); ++cfg)
      for (int64_t sp = 2; sp <= 4; ++sp) {
        const int64_t chunk = chunk_of(k, sp);
        const double t = plan_time(rounds_of(cfg, tiles_of(cfg, batch, m, n) * sp), chunk, sp, batch * m * n);
        if (t < tbest) tbest = t, best = Plan{cfg, (int)((k + chunk - 1) / chunk), chunk};
      }
  }
  // C256W from K = 2048: there its faster loop outweighs a slower start and
  // end (C256 / C256W, us: 8192 x 8192 at K = 1024 139 / 148, 1536 202 / 203,
  // 3072 376 / 364; 4096 x 12288 at K = 4096 368 / 357).
  if (best.cfg == 1 && best.splits == 1 && k >= 2048) best.cfg = 3;
  // An m-contiguous A (a weight gradient dY^T X) reads both operands through
  // transposing LDS reads, which 256x256 tiles halve per flop: it takes them
  // when they fill the CUs, or in K splits that do when C128 would leave part
  // of a single round empty (1536 x 3072 at K = 16384: 288 C128 tiles 233 us, 72
  // in three splits 160).  Splits have to save 15% by the model, which leaves
  // out the burst of the partial sums (8192 x 3072 at K = 8192: 400 us in one,
  // 433 in two).  A k-contiguous (or packed) B may take C192 below a
  // round of C256 (8027 x 1536 at K = 8192 205 us, in C128 243; 6790 x 1713 at K =
  // 4608 114 and 126).  Smaller outputs take split-K C128, with half the splits
  // (768 x 768 at K = 16384 33 / 40; 768 x 3072 is 96 / 89 by itself, but a
  // training step of such layers was 0.3 ms slower for the partial sums).
  bool planned = false;
  if (!a_kcontig && m >= 256 && n >= 256 && t128 >= kCUs) {
    const double r0 = t256 >= kCUs ? 1e30 : rounds_of(0, t128), r1 = rounds_of(1, t256);
    const double r2 = b_kcontig && t256 < kCUs && t192 >= fill ? rounds_of(2, t192) : 1e30;
    const double r = r2 < r0 && r2 < r1 ? r2 : r0 < r1 ? r0 : r1, whole = plan_time(r, k, 1, 0);
    double tbest = whole;
    best = Plan{r == r2 ? 2 : r == r0 ? 0 : k >= 2048 ? 3 : 1, 1, k};
    for (int64_t sp = 2; sp <= 4 && k / sp >= 512; ++sp) {
      const int64_t chunk = chunk_of(k, sp);
      const double t = plan_time(rounds_of(1, t256 * sp), chunk, sp, batch * m * n);
      if (t < tbest && t < 0.85 * whole) {
        tbest = t;
        best = Plan{chunk >= 2048 ? 3 : 1, (int)((k + chunk - 1) / chunk), chunk};
      }
    }
    planned = true;
  }
  // Outputs of at most two 64x64 tiles per CU: their larger tiles leave CUs idle
  // and a k-step takes its latencies, not its MFMA time (us, larger tiles against
  // C64; K = 768 unless given: 77 x 768 11.6 / 6.3, 255 x 2304 18.1 / 7.5, 512 x
  // 3072 10.6 / 8.0, 1021 x 1024 at K = 1152 20.6 / 9.3, 2048 x 768 10.8 / 7.9;
  // weight gradients 768 x 768 at K = 4096 24.2 / 19.6, 2304 x 768 at K = 2048
  // 25.1 / 19.5).  The larger tiles win where there are more tiles (4096 x 768
  // 11.4 / 12.7) or a K long enough to split over all CUs: from K = 2048 on past
  // 2.9e9 multiply-adds, counting whole tiles (264 tiles at K = 5144 27.1 / 34.9,
  // 171 at 6640 23.9 / 32.0, 294 at 2952 22.1 / 28.6, but 100 at 4096 0.88 of the
  // time), weight gradients past 3.8e9 (1024 x 1024 at K = 4096 26.0 / 27.9, 512 x
  // 2048 at K = 4096 24.3 / 27.8, 768 x 768 at K = 8192 24.1 / 27.2, 768 x 3072 at K
  // = 2048 24.5 / 26.4).
  const int64_t t64 = tiles_of(4, batch, m, n);
  const double work64 = (double)t64 * 64 * 64 * (double)k;
  if (t64 <= 2 * kCUs && (a_kcontig ? k < 2048 || work64 <= 2.9e9 : work64 <= 3.8e9))
    best = Plan{4, 1, k}, planned = false;
  static const char* forced = getenv("MI355X_GEMM_TILE");  // tuning override: "64", "128", "192", "256" or "257" (C256W)
  if (forced) {
    const double f = atof(forced);
    best.cfg = f == 256 ? 1 : (f > 256 ? 3 : (f == 192 && b_kcontig ? 2 : (f == 64 ? 4 : 0)));
    best = Plan{best.cfg, 1, k};
    planned = false;
  }
  const int64_t tiles = tiles_of(best.cfg, batch, m, n);
  if (!planned && best.splits == 1 && tiles < kCUs && k >= 2048) {
    // as many K splits as keep every block in the first round of block
    // slots: a second, partly filled round would double the time
    const int64_t slots = best.cfg == 1 || best.cfg == 3 ? kCUs : 2 * kCUs;  // block slots of the chosen config
    int64_t s = slots / tiles;
    const int64_t max_s = k / 512;
    if (s > max_s) s = max_s;
    if (s > 64) s = 64;
    if (s > 1) {
      const int64_t chunk = chunk_of(k, s), sp = (k + chunk - 1) / chunk;
      // C192 from three quarters of the CUs on: not where its partial sums cost
      // more than the second block per CU gains (2000 x 2243 at K = 2304 36.2 us,
      // 43.6 in two splits; but 4393 x 2216 at K = 2275 75.0 and 69.9)
      if (best.cfg != 2 || tiles < kCUs * 3 / 4 ||
          plan_time(rounds_of(2, tiles * sp), chunk, sp, batch * m * n) <
              1.05 * plan_time(rounds_of(2, tiles), k, 1, 0))
        best.splits = (int)sp, best.kchunk = chunk;
    }
  }
  // Over a very long K a round of C256W takes 1.4 units against the others'
  // model (50257 into 768 columns, us, before / C256W: 16384 rows C192 1386 /
  // 1268, in four splits 1211; 8192 rows C192 977 / in two splits 660; 2048 rows
  // C128 in 5 splits 204 / in ten 180).  It has to save a fifth by the model, and
  // a split to be 3072 long: four waves start and end a tile slowly (811 x 1382
  // at K = 8192 in ten splits 44.9 us, C128 in six 36.9; 4421 x 315 at K = 14518 in
  // seven 79.1, C128 in four 65.9).
  if (a_kcontig && k >= 8192 && m >= 256 && n >= 256 && best.cfg != 4 && !forced) {
    const double r = best.cfg == 3 ? 1.4 * (double)((tiles * best.splits + kCUs - 1) / kCUs)
                                   : rounds_of(best.cfg, tiles * best.splits);
    double tbest = 0.8 * plan_time(r, best.kchunk, best.splits, batch * m * n);
    const double whole = plan_time(1.4 * (double)((t256 + kCUs - 1) / kCUs), k, 1, 0);
    for (int64_t sp = 1; sp <= 10; ++sp) {
      const int64_t chunk = chunk_of(k, sp);
      const double t = plan_time(1.4 * (double)((t256 * sp + kCUs - 1) / kCUs), chunk, sp, batch * m * n);
      if (t < tbest && (sp == 1 || (t < 0.85 * whole && chunk >= 3072))) tbest = t, best = Plan{3, (int)((k + chunk - 1) / chunk), chunk};
    }
  }
  return best;
}

}  // namespace

// Sum the split-K partials into C and, with rs_slots > 0, the row-sum
// partials into the row sums; returns -1 when the C sum needs the scalar
// kernel (then the caller sums the row sums itself).
int splitk_finish(const GemmArgs& g, int64_t batch, int splits, int rs_slots, hipStream_t s) {
  const int64_t total = batch * g.m * g.n;
  const int64_t c_align = g.c_dt == MI355X_F32 ? 16 : 8;
  if (g.n % 4 == 0 && g.c_rs % 4 == 0 && g.c_bs % 4 == 0 && (uintptr_t)g.c % c_align == 0 &&
      (int64_t)splits * total < (1ll << 31)) {
    int64_t blocks = (total / 4 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (rs_slots > 0) {
      const int64_t rblocks = min((batch * g.m + 31) / 32, (int64_t)65536);
      const unsigned grid = (unsigned)(blocks + rblocks);
      switch (g.c_dt) {
        case MI355X_F32: splitk_rowsum_reduce<float><<<grid, 256, 0, s>>>(g, splits, (int)batch, rs_slots, (uint32_t)blocks); break;
        case MI355X_BF16: splitk_rowsum_reduce<bf16><<<grid, 256, 0, s>>>(g, splits, (int)batch, rs_slots, (uint32_t)blocks); break;
        default: splitk_rowsum_reduce<f16><<<grid, 256, 0, s>>>(g, splits, (int)batch, rs_slots, (uint32_t)blocks); break;
      }
      return check_launch("mi355x_gemm splitk_rowsum_reduce");
    }
    switch (g.c_dt) {
      case MI355X_F32: splitk_reduce4<float><<<(unsigned)blocks, 256, 0, s>>>(g, splits, (int)batch); break;
      case MI355X_BF16: splitk_reduce4<bf16><<<(unsigned)blocks, 256, 0, s>>>(g, splits, (int)batch); break;
      default: splitk_reduce4<f16><<<(unsigned)blocks, 256, 0, s>>>(g, splits, (int)batch); break;
    }
    return check_launch("mi355x_gemm splitk_reduce");
  }
  int64_t blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  splitk_reduce<<<(unsigned)blocks, 256, 0, s>>>(g, splits, batch);
  const int rc = check_launch("mi355x_gemm splitk_reduce");
  return rc ? rc : -1;
}

namespace {

template <typename T>
int launch_mfma(GemmArgs g, int64_t batch, const Plan& p, hipStream_t s) {
  const bool kt = g.k % 64 != 0;
  const int cfg = g.rowsum && p.cfg == 3 ? 1 : p.cfg;  // the same tiles; C256W takes no row sums
  int rc = kt ? gemm_tiles<T, true>(g, batch, cfg, p.splits, s) : gemm_tiles<T, false>(g, batch, cfg, p.splits, s);
  if (rc || !g.part) return rc;
  const int rs_slots = g.rowsum ? (int)(p.splits * rs_slots_of(p.cfg, g.n)) : 0;
  rc = splitk_finish(g, batch, p.splits, rs_slots, s);
  if (rc != -1) return rc;  // done (or failed)
  if (!g.rowsum) return MI355X_OK;
  const int64_t blocks = min((batch * g.m + 31) / 32, (int64_t)65536);
  rowsum_reduce<<<(unsigned)blocks, 256, 0, s>>>(g, (int)(p.splits * rs_slots_of(p.cfg, g.n)), batch);
  return check_launch("mi355x_gemm rowsum_reduce");
}

bool fdt(int d) { return d == MI355X_F32 || d == MI355X_BF16 || d == MI355X_F16; }

// Workspace layout of the MFMA path: [split-K partials][packed A][packed B].
struct WsLayout {
  bool pack_a, pack_b;
  int64_t kp;
  int64_t part_bytes, a_bytes, b_bytes, total;
  Plan plan;
};

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

WsLayout ws_layout(int64_t batch, int64_t m, int64_t n, int64_t k, const void* a, int64_t a_rs,
                   int64_t a_cs, int64_t a_bs, const void* b, int64_t b_rs, int64_t b_cs,
                   int64_t b_bs) {
  WsLayout w{};
  w.kp = (k + 63) / 64 * 64;
  // In place when every 16-byte load is aligned: k-contiguous operands need
  // an 8-element row stride, m/n-contiguous ones an 8-element k stride.  K
  // tails are masked in the kernel; a last partial 8-element chunk may read
  // into row padding, so the contiguous extent must be padded to 8.
  auto up8 = [](int64_t v) { return (v + 7) / 8 * 8; };
  auto in_place = [&](const void* p, int64_t rs, int64_t cs, int64_t bs, int64_t nrows) {
    if (bs % 8 != 0 || (p != nullptr && !aligned16(p))) return false;
    if (cs == 1) return rs % 8 == 0 && rs >= up8(k);
    return cs % 8 == 0 && cs >= up8(nrows);
  };
  // An m/n-contiguous operand that is small next to the product (a weight in
  // dX = dY W) is still packed: the copy costs under ~3% of the GEMM and the
  // k-contiguous fragment reads are cheaper than transposing ones.
  static const char* no_small_pack = getenv("MI355X_GEMM_NO_SMALL_PACK");  // tuning override
  // Not at k <= 1024: there one pass over the weight is a large share of the
  // GEMM, and the transposing reads cost little over so few k-steps (dX of a
  // 768-wide projection: 908 -> 977 TF/s in place).
  const double small_rows = no_small_pack || k <= 1024 ? 0.0 : 2e-4 * (double)m * (double)n;
  w.pack_a = !in_place(a, a_rs, a_cs, a_bs, m) || (a_cs != 1 && (double)m < small_rows);
  // B as [n rows][k]: row stride b_cs, k stride b_rs
  w.pack_b = !in_place(b, b_cs, b_rs, b_bs, n) || (b_rs != 1 && (double)n < small_rows);
  w.plan = plan_gemm(batch, m, n, k, w.pack_a || a_cs == 1, w.pack_b || b_rs == 1);
  auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
  // split-K partials of C, then of the optional row sums of A
  w.part_bytes = w.plan.splits > 1 ? up((int64_t)w.plan.splits * batch * m * n * 4) +
                                         up((int64_t)w.plan.splits * rs_slots_of(w.plan.cfg, n) * batch * m * 4)
                                   : 0;
  const int64_t ab = a_bs == 0 ? 1 : batch, bb = b_bs == 0 ? 1 : batch;
  w.a_bytes = w.pack_a ? up(ab * m * w.kp * 2) : 0;
  w.b_bytes = w.pack_b ? up(bb * n * w.kp * 2) : 0;
  w.total = w.part_bytes + w.a_bytes + w.b_bytes;
  return w;
}

int pack(uint16_t* dst, const void* src, int64_t batch, int64_t rows, int64_t kdim, int64_t ld,
         int64_t row_stride, int64_t k_stride, int64_t sbs, hipStream_t s) {
  // row_stride == 1: rows contiguous (transpose); else k_stride == 1 (straight)
  const bool transposed = row_stride == 1 && k_stride != 1;
  dim3 grid(ceil_div(ld, 64), ceil_div(rows, 64), (unsigned)batch);
  const int64_t stride = transposed ? k_stride : row_stride;
  const bool v8 = aligned16(src) && stride % 8 == 0 && sbs % 8 == 0 && ld % 64 == 0 &&
                  (!transposed || rows % 8 == 0);
  if (v8) {
    pack_k_contig_v8<<<grid, 256, 0, s>>>(dst, ld, rows * ld, (const uint16_t*)src, stride, sbs, rows, kdim,
                                          transposed ? 1 : 0);
    return check_launch("mi355x_gemm pack");
  }
  pack_k_contig<<<grid, 256, 0, s>>>(dst, ld, rows * ld, (const uint16_t*)src,
                                      transposed ? k_stride : row_stride, sbs, rows, kdim,
                                      transposed ? 1 : 0);
  return check_launch("mi355x_gemm pack");
}

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" int64_t mi355x_gemm_workspace_bytes(const void* a, int64_t a_rs, int64_t a_cs,
                                               int64_t a_bs, const void* b, int64_t b_rs,
                                               int64_t b_cs, int64_t b_bs, int ab_dtype,
                                               int64_t batch, int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  if (ab_dtype == MI355X_F32) return gemm_f32_workspace(batch, m, n, k);
  return ws_layout(batch, m, n, k, a, a_rs, a_cs, a_bs, b, b_rs, b_cs, b_bs).total;
}

extern "C" int mi355x_gemm_ex(void* c, int c_dtype, int64_t c_rs, int64_t c_bs, const void* a,
                              int64_t a_rs, int64_t a_cs, int64_t a_bs, const void* b, int64_t b_rs,
                              int64_t b_cs, int64_t b_bs, int ab_dtype, const void* bias,
                              int bias_dtype, int flags, void* a_rowsum, int a_rowsum_dtype,
                              int64_t batch, int64_t m, int64_t n, int64_t k, void* workspace,
                              int64_t ws_bytes, mi355x_stream_t stream) {
  MI_REQUIRE(fdt(ab_dtype) && fdt(c_dtype), "mi355x_gemm: unsupported dtype");
  MI_REQUIRE(!bias || fdt(bias_dtype), "mi355x_gemm: unsupported bias dtype");
  MI_REQUIRE(!a_rowsum || fdt(a_rowsum_dtype), "mi355x_gemm: unsupported row-sum dtype");
  MI_REQUIRE((flags & ~(MI355X_GEMM_BETA | MI355X_GEMM_ROUND)) == 0, "mi355x_gemm: unknown flags %d", flags);
  const int beta = (flags & MI355X_GEMM_BETA) ? 1 : 0;
  const int round_c = (flags & MI355X_GEMM_ROUND) ? 1 : 0;
  MI_REQUIRE(!(beta && round_c), "mi355x_gemm: ROUND cannot be combined with BETA");
  MI_REQUIRE(batch >= 1 && m >= 0 && n >= 0 && k >= 0, "mi355x_gemm: bad shape");
  MI_REQUIRE(batch < 65536 && m < (1ll << 31) && n < (1ll << 31), "mi355x_gemm: shape too large");
  if (m == 0 || n == 0) return MI355X_OK;
  MI_REQUIRE(k > 0, "mi355x_gemm: k == 0 must be handled by the caller");
  MI_REQUIRE(a_rs == 1 || a_cs == 1, "mi355x_gemm: A needs a unit row or column stride");
  MI_REQUIRE(b_rs == 1 || b_cs == 1, "mi355x_gemm: B needs a unit row or column stride");
  MI_REQUIRE(c && a && b, "mi355x_gemm: null pointer");
  hipStream_t s = (hipStream_t)stream;
  GemmArgs g{c, c_dtype, c_rs, c_bs, a, a_rs, a_cs, a_bs, b, b_rs, b_cs, b_bs, bias, bias_dtype,
             beta, m, n, k, nullptr, k, 1, 1, 1, ab_dtype, round_c, a_rowsum, a_rowsum_dtype, nullptr};
  if (ab_dtype == MI355X_F32) {
    MI_REQUIRE(!a_rowsum && !round_c, "mi355x_gemm: row sums and ROUND need 16-bit operands");
    return gemm_f32_launch(g, batch, workspace, ws_bytes, s);
  }
  WsLayout w = ws_layout(batch, m, n, k, a, a_rs, a_cs, a_bs, b, b_rs, b_cs, b_bs);
  MI_REQUIRE(batch * w.plan.splits < 65536, "mi355x_gemm: batch x splits too large");
  MI_REQUIRE(tiles_of(w.plan.cfg, 1, m, n) < (1ll << 31), "mi355x_gemm: shape too large");
  // the epilogue addresses a tile with 32-bit offsets: 256 rows of C (or of
  // the n-wide split-K partials) must span less than 2^31 elements
  MI_REQUIRE(c_rs < (1ll << 22) && n < (1ll << 22), "mi355x_gemm: C row stride too large");
  if (w.total > 0 && (!workspace || ws_bytes < w.total))
    return fail(MI355X_EWORKSPACE, "mi355x_gemm: workspace %lld < %lld", (long long)ws_bytes,
                (long long)w.total);
  char* ws = (char*)workspace;
  if (w.pack_a) {
    uint16_t* pa = (uint16_t*)(ws + w.part_bytes);
    const int64_t nb = a_bs == 0 ? 1 : batch;
    int rc = pack(pa, a, nb, m, k, w.kp, a_rs, a_cs, a_bs, s);
    if (rc) return rc;
    g.a = pa; g.a_rs = w.kp; g.a_cs = 1; g.a_bs = a_bs == 0 ? 0 : m * w.kp;
  }
  if (w.pack_b) {
    uint16_t* pb = (uint16_t*)(ws + w.part_bytes + w.a_bytes);
    const int64_t nb = b_bs == 0 ? 1 : batch;
    // B viewed as [n rows][k]: row stride b_cs, k stride b_rs
    int rc = pack(pb, b, nb, n, k, w.kp, b_cs, b_rs, b_bs, s);
    if (rc) return rc;
    g.b = pb; g.b_rs = 1; g.b_cs = w.kp; g.b_bs = b_bs == 0 ? 0 : n * w.kp;
  }
  // packed operands are zero-padded to kp; the kernel masks k >= K
  if (w.plan.splits > 1) {
    g.part = (float*)ws;
    g.kchunk = w.plan.kchunk;
    g.rs_part = (float*)(ws + (((int64_t)w.plan.splits * batch * m * n * 4 + 255) / 256 * 256));
  }
  if (ab_dtype == MI355X_BF16) return launch_mfma<bf16>(g, batch, w.plan, s);
  return launch_mfma<f16>(g, batch, w.plan, s);
}

extern "C" int mi355x_gemm(void* c, int c_dtype, int64_t c_rs, int64_t c_bs, const void* a,
                           int64_t a_rs, int64_t a_cs, int64_t a_bs, const void* b, int64_t b_rs,
                           int64_t b_cs, int64_t b_bs, int ab_dtype, const void* bias,
                           int bias_dtype, int beta, int64_t batch, int64_t m, int64_t n,
                           int64_t k, void* workspace, int64_t ws_bytes, mi355x_stream_t stream) {
  return mi355x_gemm_ex(c, c_dtype, c_rs, c_bs, a, a_rs, a_cs, a_bs, b, b_rs, b_cs, b_bs, ab_dtype, bias,
                        bias_dtype, beta ? MI355X_GEMM_BETA : 0, nullptr, 0, batch, m, n, k, workspace,
                        ws_bytes, stream);
}
