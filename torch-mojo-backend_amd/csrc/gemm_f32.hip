// GEMM with f32 operands on v_mfma_f32_16x16x4_f32 (f32 products and sums, as
// a chain of FMAs; 256 flops per clock and CU, 157 TFLOP/s nominal).
//
// A short K over a large output runs on plain FMAs instead (takes_fma).
//
// Bound: the MFMA rate.  One MFMA takes 32 cycles and two operand registers,
// so LDS and L2 traffic are small next to it at a 64x64 wave tile (8 16-byte
// LDS reads per 64 MFMAs); what has to be kept off its path is load latency
// (two stages of direct global -> LDS loads, two blocks per CU) and idle CUs
// (the tile and split-K rule in plan_f32).
//
// Only the pairing of k between A and B matters, so within a 16-k slab lane
// group g holds k = 4g .. 4g+3 and MFMA j multiplies the k = 4g + j:
//   k-contiguous operand: tile [row][32 k], 16-byte chunks XOR-swizzled by
//     (row >> 1) & 7; one 16-byte read is a fragment's operand for 4 MFMAs;
//   m/n-contiguous operand: tile [k][rows]; one read of F consecutive rows at
//     one k is one operand of F fragments, so fragment i holds rows F*r + i.
// k-contiguous tiles hold their rows in that order too, so a lane's results
// are F adjacent columns of C and leave in one store (16384 x 3072 x 768 with
// both operands k-contiguous: 705 -> 655 us, 118 TFLOP/s; n-contiguous B
// 127 TFLOP/s).
// VEC loads tiles 16 bytes per lane, which needs 16-byte aligned rows and a
// contiguous extent that is a multiple of 4; other operands are loaded 4
// bytes per lane into the same tiles (still an eighth of the MFMA time).
#include "common.h"
#include "gemm.h"
#include "mfma.h"

extern __shared__ __attribute__((aligned(16))) char gemm_f32_smem[];

namespace mi {
namespace {

constexpr int kCUs = 256;
constexpr int kBK = 32;   // k per stage
constexpr int kNT = 256;  // 4 waves, 2 x 2

__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
constexpr int kCPR = kBK / 4;  // 16-byte chunks per k-contiguous row

// Row of the operand at row p of a k-contiguous tile: within each wave's
// F fragments, row F * r + i lies at 16 i + r, so that fragment i holds rows
// F * r + i as with an m/n-contiguous operand and a lane's results are
// adjacent columns of C.
template <int F>
__device__ __forceinline__ int src_row(int p) { return p / (16 * F) * (16 * F) + (p & 15) * F + (p / 16) % F; }

// Loads a ROWS x 32-k tile of an operand that is contiguous in k.
template <int ROWS, bool VEC>
struct LoadK {
  static constexpr int RPI = VEC ? 64 / kCPR : 64 / kBK;  // rows per wave instruction
  static constexpr int F = ROWS / 32;
  static constexpr int ITERS = ROWS / (RPI * 4);      // instructions per wave
  const float* src[VEC ? ITERS : 1];
  const float* base;
  int64_t ld, row0, rows;
  int kof;

  __device__ __forceinline__ void init(const float* b, int64_t ld_, int64_t r0, int64_t n) {
    const int lane = threadIdx.x & 63, wave = wave_id();
    if constexpr (VEC) {
      // swz repeats every 16 rows and a wave's instructions are 32 rows
      // apart, so a lane's chunk is the same for all of them
      const int r = wave * RPI + lane / kCPR;
      kof = ((lane % kCPR) ^ swz(r)) * 4;
#pragma unroll
      for (int it = 0; it < ITERS; ++it) src[it] = b + min(r0 + src_row<F>(r + it * RPI * 4), n - 1) * ld_;
    } else {
      base = b, ld = ld_, row0 = r0, rows = n;
    }
  }
  __device__ __forceinline__ void issue(int64_t k0, int64_t kend, char* dst) const {
    const unsigned lds = lds_base_of(dst) + wave_id() * (VEC ? 1024 : 256);
    if constexpr (VEC) {
      const int64_t k = k0 + kof < kend ? k0 + kof : k0;  // past the end: masked later
#pragma unroll
      for (int it = 0; it < ITERS; ++it) dma_b128(src[it] + k, lds + it * 4096);
    } else {
      const int lane = threadIdx.x & 63;
#pragma unroll 4
      for (int it = 0; it < ITERS; ++it) {
        const int r = (it * 4 + wave_id()) * RPI + lane / kBK, p = lane % kBK;
        const int64_t k = k0 + (((p >> 2) ^ swz(r)) << 2) + (p & 3);
        dma_b32(base + min(row0 + src_row<F>(r), rows - 1) * ld + (k < kend ? k : k0), lds + it * 1024);
      }
    }
  }
};

// Loads a 32-k x ROWS tile of an operand that is contiguous in its rows.
template <int ROWS, bool VEC>
struct LoadMN {
  static constexpr int EPI = VEC ? 256 : 64;          // floats per wave instruction
  static constexpr int ITERS = kBK * ROWS / (EPI * 4);
  const float* base;
  int64_t ld;
  int64_t col[VEC || ROWS == 64 ? 1 : 2];
  static constexpr int NCOL = VEC || ROWS == 64 ? 1 : 2;  // 64-float halves of a k-row

  __device__ __forceinline__ void init(const float* b, int64_t ld_, int64_t r0, int64_t n) {
    const int lane = threadIdx.x & 63;
    base = b, ld = ld_;
    if constexpr (VEC) {
      const int64_t c = r0 + (lane % (ROWS / 4)) * 4;
      col[0] = c < n ? c : n - 4;
    } else {
#pragma unroll
      for (int h = 0; h < NCOL; ++h) col[h] = min(r0 + h * 64 + lane, n - 1);
    }
  }
  __device__ __forceinline__ void issue(int64_t k0, int64_t kend, char* dst) const {
    const int lane = threadIdx.x & 63, wave = wave_id();
    const unsigned lds = lds_base_of(dst) + wave * (EPI * 4);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int q = it * 4 + wave;  // instruction q holds floats [q * EPI, (q + 1) * EPI) of the tile
      if constexpr (VEC) {
        const int64_t k = min(k0 + q * (EPI / ROWS) + lane / (ROWS / 4), kend - 1);
        dma_b128(base + k * ld + col[0], lds + it * (EPI * 16));
      } else {
        const int64_t k = min(k0 + q / NCOL, kend - 1);
        int64_t c = col[0];
        if constexpr (NCOL == 2) c = (wave & 1) ? col[1] : col[0];  // q and wave have one parity
        dma_b32(base + k * ld + c, lds + it * (EPI * 16));
      }
    }
  }
};

template <int ROWS, bool K_CONTIG, bool VEC>
struct Load : LoadK<ROWS, VEC> {};
template <int ROWS, bool VEC>
struct Load<ROWS, false, VEC> : LoadMN<ROWS, VEC> {};

// The operands f[i] (fragments i, MFMAs j = 0..3) of one 16-k slab.
template <int ROWS, bool K_CONTIG, int F>
__device__ __forceinline__ void frags(const char* tile, int r0, int ks, float (&f)[F][4]) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  if constexpr (K_CONTIG) {
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int r = r0 + i * 16 + lr;
      const f32x4 v = *(const f32x4*)(tile + r * (kBK * 4) + (((ks * 4 + lg) ^ swz(r)) << 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) f[i][j] = v[j];
    }
  } else {
    typedef float vec __attribute__((ext_vector_type(F)));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const vec v = *(const vec*)(tile + ((ks * 16 + 4 * lg + j) * ROWS + r0 + F * lr) * 4);
#pragma unroll
      for (int i = 0; i < F; ++i) f[i][j] = v[i];
    }
  }
}

template <int F>
__device__ __forceinline__ void mask(float (&f)[F][4], int64_t k, int64_t kend) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (k + j >= kend)
#pragma unroll
      for (int i = 0; i < F; ++i) f[i][j] = 0.f;
}

// TILE x TILE of C per block, a quarter (two by two) per wave.  M_FIRST: the
// tiles of one column of C are neighbours in the block order.
template <int TILE, bool A_K, bool B_K, bool VEC>
__global__ void __launch_bounds__(kNT, 2) gemm_f32_tile(GemmArgs g, int tiles_m, int m_first) {
  constexpr int W = TILE / 2, F = W / 16;
  constexpr int HALF = TILE * kBK * 4, STAGE = 2 * HALF;
  char* const lds = gemm_f32_smem;

  // Each XCD takes a contiguous run of the (split, batch)-major tile list (the
  // hardware deals blocks to the 8 XCDs round robin), so its blocks share
  // panels in its L2.
  const uint32_t nt = gridDim.x, total = nt * gridDim.y;
  uint32_t L = blockIdx.x + nt * blockIdx.y;
  {
    const uint32_t xcd = L & 7, q = total >> 3, r = total & 7;
    L = xcd * q + min(xcd, r) + (L >> 3);
  }
  const uint32_t plane = L / nt, t = L - plane * nt;
  uint32_t tm, tn;
  if (m_first) tn = t / (uint32_t)tiles_m, tm = t - tn * (uint32_t)tiles_m;
  else tm = t / (uint32_t)g.tiles_n, tn = t - tm * (uint32_t)g.tiles_n;
  const uint32_t split = plane / (uint32_t)g.batch, bidx = plane - split * (uint32_t)g.batch;
  const int64_t m0 = (int64_t)tm * TILE, n0 = (int64_t)tn * TILE;
  int64_t kbeg = 0, kend = g.k;
  if (g.part) kbeg = (int64_t)split * g.kchunk, kend = min(g.k, kbeg + g.kchunk);

  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wm = wave_id() >> 1, wn = wave_id() & 1;
  Load<TILE, A_K, VEC> la;
  Load<TILE, B_K, VEC> lb;
  la.init((const float*)g.a + bidx * g.a_bs, A_K ? g.a_rs : g.a_cs, m0, g.m);
  lb.init((const float*)g.b + bidx * g.b_bs, B_K ? g.b_cs : g.b_rs, n0, g.n);

  f32x4 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  la.issue(kbeg, kend, lds);
  lb.issue(kbeg, kend, lds + HALF);
  int cur = 0;
  for (int64_t k0 = kbeg; k0 < kend; k0 += kBK, cur ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this stage has landed
    __syncthreads();
    const char* at = lds + cur * STAGE;
    const char* bt = at + HALF;
    // All of the stage's operands are read before its MFMAs, and the next
    // stage's loads are issued in the shadow of the first reads: one LDS
    // latency a stage.
    float a[kBK / 16][F][4], b[kBK / 16][F][4];
    frags<TILE, A_K, F>(at, wm * W, 0, a[0]);
    frags<TILE, B_K, F>(bt, wn * W, 0, b[0]);
    if (k0 + kBK < kend) {  // into the stage that every wave has finished reading
      la.issue(k0 + kBK, kend, lds + (cur ^ 1) * STAGE);
      lb.issue(k0 + kBK, kend, lds + (cur ^ 1) * STAGE + HALF);
    }
#pragma unroll
    for (int ks = 1; ks < kBK / 16; ++ks) {
      frags<TILE, A_K, F>(at, wm * W, ks, a[ks]);
      frags<TILE, B_K, F>(bt, wn * W, ks, b[ks]);
    }
    if (k0 + kBK > kend) {  // both operands: what lies past the end may be inf or NaN
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        const int64_t k = k0 + ks * 16 + 4 * lg;
        mask(a[ks], k, kend);
        mask(b[ks], k, kend);
      }
    }
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ks][i][s], b[ks][j][s], acc[i][j], 0, 0, 0);
  }

  // lane (lg, lr) holds rows 4 lg + e of fragment row i and column lr of
  // fragment column j, permuted as the operand was read
  const int64_t row0 = m0 + wm * W, col0 = n0 + wn * W;
  float bias[F];
  int64_t cols[F];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    cols[j] = col0 + F * lr + j;
    bias[j] = (!g.part && g.bias && cols[j] < g.n) ? ld_any(g.bias, g.bias_dt, cols[j]) : 0.f;
  }
  float* P = nullptr;
  int64_t rs = g.c_rs;
  if (g.part) P = g.part + ((int64_t)split * g.batch + bidx) * g.m * g.n, rs = g.n;
  else if (g.c_dt == MI355X_F32) P = (float*)g.c + bidx * g.c_bs;
  char* Cb = (char*)g.c + bidx * g.c_bs * 2;  // 16-bit C
  const bool beta = g.beta && !g.part;
  // F adjacent columns per lane leave in one store, which the hardware splits
  // where it is not aligned
  struct Out { float v[F]; };
  const bool wide = P && !beta && cols[F - 1] < g.n;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t row = row0 + F * (4 * lg + e) + i;
      if (row >= g.m) continue;
      if (wide) {
        Out out;
#pragma unroll
        for (int j = 0; j < F; ++j) out.v[j] = acc[i][j][e] + bias[j];
        *(Out*)(P + row * rs + cols[0]) = out;
        continue;
      }
#pragma unroll
      for (int j = 0; j < F; ++j) {
        if (cols[j] >= g.n) continue;
        const int64_t off = row * rs + cols[j];
        float v = acc[i][j][e] + bias[j];
        if (P) P[off] = beta ? v + P[off] : v;
        else st_any(Cb, g.c_dt, off, beta ? v + ld_any(Cb, g.c_dt, off) : v);
      }
    }
}

// 64x64 tile by FMAs, 4x4 outputs per thread, in stages of 16 k.
__global__ void __launch_bounds__(256) gemm_f32_fma(GemmArgs g) {
  __shared__ float As[16][64 + 4];
  __shared__ float Bs[16][64 + 4];
  const int64_t batch = blockIdx.z;
  const int64_t m0 = (int64_t)blockIdx.y * 64, n0 = (int64_t)blockIdx.x * 64;
  const float* A = (const float*)g.a + batch * g.a_bs;
  const float* B = (const float*)g.b + batch * g.b_bs;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  float acc[4][4] = {};
  for (int64_t k0 = 0; k0 < g.k; k0 += 16) {
    for (int e = threadIdx.x; e < 16 * 64; e += 256) {
      const int kk = e / 64, r = e % 64;
      const int64_t gm = m0 + r, gk = k0 + kk, gn = n0 + r;
      As[kk][r] = (gm < g.m && gk < g.k) ? A[gm * g.a_rs + gk * g.a_cs] : 0.f;
      Bs[kk][r] = (gn < g.n && gk < g.k) ? B[gk * g.b_rs + gn * g.b_cs] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i], b[i] = Bs[kk][tx * 4 + i];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
    }
    __syncthreads();
  }
  void* Cb = (char*)g.c + batch * g.c_bs * (g.c_dt == MI355X_F32 ? 4 : 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t row = m0 + ty * 4 + i;
    if (row >= g.m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t col = n0 + tx * 4 + j;
      if (col >= g.n) continue;
      float v = acc[i][j] + (g.bias ? ld_any(g.bias, g.bias_dt, col) : 0.f);
      const int64_t off = row * g.c_rs + col;
      if (g.beta) v += ld_any(Cb, g.c_dt, off);
      st_any(Cb, g.c_dt, off, v);
    }
  }
}

// Where the FMA kernel is the faster one: up to half of its first stage, and all
// of it while there are few tiles or thin ones (matrix cores over FMA, geometric
// means of drawn shapes: up to 256 tiles 1.05 at K <= 2, 1.0 at 9 .. 16; up to 2048
// 1.33 and 1.14 .. 1.22; 14008 x 1151 at K = 1 26.8 us, on matrix cores 34.9; past
// 2048 tiles at K = 9 .. 16 0.82 .. 0.98); and many tiles of few rows or columns
// where its stages of 16 k cover K more closely than those of 32 (28 batches of 1 x
// 50257 at K = 40 121 us, on matrix cores 187, 4 x 14257 x 2 at K = 41 10.3 and 13.0;
// up to 32 rows at K = 33 .. 48 FMA takes 0.77 .. 0.91 of the time, at 49 .. 64 1.0
// .. 1.2).
bool takes_fma(int64_t batch, int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + 63) / 64) * ((n + 63) / 64) * batch, least = m < n ? m : n;
  if (least <= 32 && tiles >= 3 * kCUs) return k <= 48 || (least <= 16 && k > 64 && k <= 80);
  return k <= 8 || (k <= 16 && (tiles <= 2048 || least <= 160));
}

struct PlanF32 {
  int tile;  // 128 or 64
  int splits;
  int64_t kchunk;
};

// The tile size and the number of K splits with the least estimated time: the
// rounds of 256 CUs (blocks that share a CU share its matrix units) times a
// block's time at the rate that one block per CU was measured at (4096 x 3072,
// K = 768: 128 tiles in 3 rounds 181 us, 64 tiles in 12 rounds 208 us), plus,
// with splits, the summing launch (the partials of 4096 x 768 in 3 splits:
// 8 us).
PlanF32 plan_f32(int64_t batch, int64_t m, int64_t n, int64_t k) {
  PlanF32 best{128, 1, k};
  double tbest = 1e30;
  for (int tile = 128; tile >= 64; tile -= 64) {
    const int64_t tiles = ((m + tile - 1) / tile) * ((n + tile - 1) / tile) * batch;
    // one round of 128 tiles over a short K: a block's start and end take its time
    // (3906 x 1019 at K = 63 21.3 us, in 64 tiles 15.3)
    if (tile == 128 && k <= 64 && tiles <= kCUs) continue;
    if (tile == 64 && tiles >= 1 << 24) continue;  // a launch takes fewer than 2^32 threads
    const double per_k = 2.0 * tile * tile / (tile == 128 ? 440e3 : 375e3);  // us
    for (int64_t sp = 1; sp <= 32 && (sp == 1 || (k / sp >= 128 && tiles < 4 * kCUs)); ++sp) {
      int64_t chunk = (k + sp - 1) / sp;
      chunk = (chunk + kBK - 1) / kBK * kBK;
      const int64_t s = (k + chunk - 1) / chunk;
      if (s != sp) continue;  // the same split as a smaller sp
      const double rounds = (double)((tiles * s + kCUs - 1) / kCUs);
      double t = rounds * per_k * (double)(s > 1 ? chunk : k);
      if (s > 1) t += 3.0 + (double)(s + 1) * 4.0 * (double)(batch * m * n) / 6e6;
      if (t < tbest * 0.98) tbest = t, best = PlanF32{tile, (int)s, s > 1 ? chunk : k};
    }
  }
  return best;
}

template <int TILE, bool A_K, bool B_K, bool VEC>
int launch(const GemmArgs& g, int tiles_m, dim3 grid, hipStream_t s) {
  constexpr size_t lds = 2 * 2 * (size_t)TILE * kBK * 4;  // 64 KB at most
  size_t bytes = lds;
  if (TILE == 128 && VEC) {
    // Two blocks fit a CU.  When the last pair of rounds has only one block
    // per CU to give, the CUs whose two blocks end together take two again
    // while others idle; with the LDS of one block per CU the rounds are whole
    // (4096 x 3072, K = 768, 768 blocks: 221 -> 181 us; with more rounds two
    // per CU are faster, 1024 x 50257: 760 against 831 us, and with 4-byte
    // loads, whose latency a second block hides, K = 50257: 995 against 1093).
    const int64_t blocks = (int64_t)grid.x * grid.y;
    if (blocks <= 4 * kCUs && (blocks + kCUs - 1) / kCUs < 2 * ((blocks + 2 * kCUs - 1) / (2 * kCUs))) {
      constexpr int alone = 88 * 1024;  // more than half of a CU's 160 KB
      static const bool ok = hipFuncSetAttribute((const void*)gemm_f32_tile<TILE, A_K, B_K, VEC>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, alone) == hipSuccess;
      if (!ok) return fail(MI355X_ELAUNCH, "mi355x_gemm: cannot reserve %d bytes of LDS", alone);
      bytes = alone;
    }
  }
  gemm_f32_tile<TILE, A_K, B_K, VEC><<<grid, kNT, bytes, s>>>(g, tiles_m, tiles_m <= g.tiles_n ? 1 : 0);
  return check_launch("mi355x_gemm");
}

template <int TILE, bool VEC>
int launch_layout(const GemmArgs& g, int tiles_m, dim3 grid, hipStream_t s) {
  const bool ak = g.a_cs == 1, bk = g.b_rs == 1;
  if (ak && bk) return launch<TILE, true, true, VEC>(g, tiles_m, grid, s);
  if (ak) return launch<TILE, true, false, VEC>(g, tiles_m, grid, s);
  if (bk) return launch<TILE, false, true, VEC>(g, tiles_m, grid, s);
  return launch<TILE, false, false, VEC>(g, tiles_m, grid, s);
}

// 16-byte loads: aligned base, row and batch strides; contiguous extent and K
// multiples of 4, so that no 16 bytes straddle an end.
bool vec_ok(const void* p, int64_t ld, int64_t bs, int64_t extent) {
  return ((uintptr_t)p & 15) == 0 && ld % 4 == 0 && bs % 4 == 0 && extent % 4 == 0;
}

}  // namespace

int64_t gemm_f32_workspace(int64_t batch, int64_t m, int64_t n, int64_t k) {
  if (takes_fma(batch, m, n, k)) return 0;
  const PlanF32 p = plan_f32(batch, m, n, k);
  return p.splits > 1 ? (int64_t)p.splits * batch * m * n * 4 : 0;
}

int gemm_f32_launch(GemmArgs g, int64_t batch, void* workspace, int64_t ws_bytes, hipStream_t s) {
  if (takes_fma(batch, g.m, g.n, g.k)) {
    gemm_f32_fma<<<dim3(ceil_div(g.n, 64), ceil_div(g.m, 64), (unsigned)batch), kNT, 0, s>>>(g);
    return check_launch("mi355x_gemm");
  }
  PlanF32 p = plan_f32(batch, g.m, g.n, g.k);
  if (p.splits > 1 && (!workspace || ws_bytes < (int64_t)p.splits * batch * g.m * g.n * 4))
    p.splits = 1, p.kchunk = g.k;
  const int64_t tiles_m = (g.m + p.tile - 1) / p.tile, tiles_n = (g.n + p.tile - 1) / p.tile;
  MI_REQUIRE(batch * p.splits < 65536 && tiles_m * tiles_n * batch * p.splits < (1ll << 31),
             "mi355x_gemm: shape too large");
  g.tiles_n = (int)tiles_n;
  g.batch = (int)batch;
  g.kchunk = p.kchunk;
  g.part = p.splits > 1 ? (float*)workspace : nullptr;
  const bool vec = vec_ok(g.a, g.a_cs == 1 ? g.a_rs : g.a_cs, g.a_bs, g.a_cs == 1 ? g.k : g.m) &&
                   vec_ok(g.b, g.b_rs == 1 ? g.b_cs : g.b_rs, g.b_bs, g.b_rs == 1 ? g.k : g.n);
  const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)(batch * p.splits));
  int rc;
  if (p.tile == 128)
    rc = vec ? launch_layout<128, true>(g, (int)tiles_m, grid, s) : launch_layout<128, false>(g, (int)tiles_m, grid, s);
  else
    rc = vec ? launch_layout<64, true>(g, (int)tiles_m, grid, s) : launch_layout<64, false>(g, (int)tiles_m, grid, s);
  if (rc || !g.part) return rc;
  rc = splitk_finish(g, batch, p.splits, 0, s);
  return rc == -1 ? MI355X_OK : rc;
}

}  // namespace mi
