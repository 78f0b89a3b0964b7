// GEMM: C[b] = A[b] * B[b] (+ bias row) (+ C if beta), f32 accumulation.
//
// bf16/f16 inputs run on MFMA (v_mfma_f32_16x16x32_*).  One kernel template
// covers every layout of the training GEMMs:
//   fwd  x*W^T : A k-contiguous, B k-contiguous (W rows)
//   dX   dY*W  : A k-contiguous, B n-contiguous
//   dW   dY^T*X: A m-contiguous, B n-contiguous
// Operand tiles (64 k per step) go global -> LDS directly with
// global_load_lds_dwordx4 (each wave instruction fills 1 KB, lane i writing
// bytes [16i, 16i+16)), two stages deep: the next step's loads are issued
// right after the barrier and stream in under the current step's MFMAs.
//   k-contiguous tile: [row][64 k] rows of 128 bytes, 16-byte chunks
//     XOR-swizzled by (row >> 1) & 7 so a fragment read of 16 rows hits 16
//     distinct bank groups;
//   m/n-contiguous tile: [k][rows] with chunks swizzled by kswz(k); fragments
//     are read transposed with ds_read_b64_tr_b16.
// A lane's global source address is chosen so that its fixed LDS slot
// receives the swizzled chunk, so staging costs no registers.
//
// Block configurations (waves arranged WGM x WGN, each wave owning a
// (BM/WGM) x (BN/WGN) sub-tile of 16x16 MFMA tiles):
//   C128: 128x128, 4 waves of 64x64, 64 KB LDS, two blocks per CU;
//   C192: 128x192, 4 waves of 64x96, 80 KB LDS, two blocks per CU (B
//         k-contiguous only); N = 768, 2304, 3072 split into whole rounds;
//   C256: 256x256, 8 waves of 128x64, 128 KB LDS, one block per CU (fewer
//         LDS bytes per flop; preferred when its tiles fill the CUs evenly);
//   C256W: 256x256, 4 waves of 128x128, 160 KB LDS, one block per CU, from
//         K = 2048 where C256 would be taken;
//   C64: 64x64, 4 waves of 32x32, for outputs too small to fill the CUs
//         otherwise (one GPT-2 layer of a 77-token prompt: 11.8 -> 6.4 us a
//         product).
// The block -> tile map is XCD-aware (the hardware deals workgroups to the 8
// XCDs round-robin): each XCD walks a contiguous run of tiles, so the blocks
// sharing an L2 share operand panels.  Index math is 32-bit and the edge
// clamps are folded into per-thread base pointers once, so the prologue
// stays short next to a K = 768 main loop.
#pragma once
#include <type_traits>

#include "common.h"
#include "gemm.h"
#include "mfma.h"

extern __shared__ __attribute__((aligned(16))) char gemm_smem[];

namespace mi {
namespace {

// Row swizzle of a k-contiguous tile with 128-byte rows (64 k): row r stores its
// 16-byte chunk c in slot c ^ rswz(r).  A fragment read (16 rows at one chunk)
// then covers every bank once: 8 chunks, rows paired by (r >> 1).
__device__ __forceinline__ int rswz(int r) { return (r >> 1) & 7; }

// k-contiguous operand tile: ROWS rows x BK k, loaded by NT threads, one
// 1 KB instruction per RPI rows.  Thread (wave w, lane l) handles rows
// r = RPI*(it*WAVES + w) + l/CPR; with WAVES even the swizzled chunk of its
// slot, (l % CPR) ^ rswz(r), is the same for every `it`.  Rows past the
// operand's end reload its last row (their results are never stored).
template <int ROWS, int NT, int BK>
struct TileLoad {
  static_assert(BK == 64, "rswz");
  static constexpr int CPR = BK / 8;    // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;  // rows per 1 KB instruction
  static constexpr int WAVES = NT / 64;
  static constexpr int ITERS = ROWS / (RPI * WAVES);
  static_assert(WAVES % 2 == 0 && ITERS * RPI * WAVES == ROWS, "tile/thread mismatch");
  const char* src[ITERS];  // row base + this lane's chunk, at k = 0
  int chunk;

  __device__ __forceinline__ void init(const char* base, int64_t ld_bytes, int64_t row0, int64_t rows) {
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int r = wave * RPI + lane / CPR;
    chunk = (lane % CPR) ^ rswz(r);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      int64_t row = row0 + r + it * RPI * WAVES;
      if (row > rows - 1) row = rows - 1;
      src[it] = base + row * ld_bytes + chunk * 16;
    }
  }
  // KT: the K range may end inside this BK slab; a chunk starting past
  // kend_bytes reloads chunk 0 (masked out of the MFMAs, address valid).
  template <bool KT>
  __device__ __forceinline__ void issue(int64_t k0_bytes, char* dst, int64_t kend_bytes) const {
    const int64_t koff = (KT && k0_bytes + chunk * 16 >= kend_bytes) ? k0_bytes - chunk * 16 : k0_bytes;
    // one scalar LDS base per call; each instruction's slot is a constant offset
    const unsigned lds0 = lds_base_of(dst) + wave_id() * 1024;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) dma_b128(src[it] + koff, lds0 + it * WAVES * 1024);
  }
  template <bool KT>
  __device__ __forceinline__ void issue_range(int64_t k0_bytes, char* dst, int64_t kend_bytes, int lo, int hi) const {
    const int64_t koff = (KT && k0_bytes + chunk * 16 >= kend_bytes) ? k0_bytes - chunk * 16 : k0_bytes;
    const unsigned lds0 = lds_base_of(dst) + wave_id() * 1024;
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
      if (it >= lo && it < hi) dma_b128(src[it] + koff, lds0 + it * WAVES * 1024);
  }
};

// m/n-contiguous operand tile: BK k-rows of ROWS elements, 16-byte chunks
// XOR-swizzled by s(k) = 2 * ((k & 3) | ((k >> 1) & 4)).  A transposing
// fragment read serves each half-wave from 8 k-rows x 2 adjacent chunks
// (c, c ^ 1); s takes 8 distinct even values on those k-rows, so the 16
// (k-row, chunk) pairs land on 16 distinct 16-byte bank groups.
// 64-element rows (8 chunks, 32 banks) leave a bank to every other k-row, so
// there s takes 4 distinct even values on the 4 k-rows of one parity.
template <int CPR>
__device__ __forceinline__ int kswz(int k) {
  return CPR >= 16 ? 2 * ((k & 3) | ((k >> 1) & 4)) : 2 * (((k >> 1) & 1) | ((k >> 2) & 2));
}

template <int ROWS, int NT, int BK>
struct TileLoadT {
  static constexpr int ROWB = ROWS * 2;
  static constexpr int CPR = ROWS / 8;     // chunks per k-row
  static constexpr int KPI = 1024 / ROWB;  // k-rows per 1 KB instruction
  static constexpr int WAVES = NT / 64;
  static constexpr int ITERS = BK / KPI / WAVES;
  static_assert(CPR >= 8 && ITERS * KPI * WAVES == BK, "tile/thread mismatch");
  const char* base;
  int64_t ld;              // bytes between k-rows
  int64_t col_off[ITERS];  // byte offset of this lane's (clamped) chunk
  int kr[ITERS];           // this lane's k-row within the slab

  // A last partial chunk of rows reads into the row padding (the k stride
  // is at least the row count rounded up to 8, checked by the caller).
  __device__ __forceinline__ void init(const char* b, int64_t ld_bytes, int64_t r0, int64_t rows) {
    const int lane = threadIdx.x & 63, wave = wave_id();
    base = b;
    ld = ld_bytes;
    const int64_t last_chunk = ((rows - 1) >> 3) << 3;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      kr[it] = (it * WAVES + wave) * KPI + lane / CPR;
      int64_t m = r0 + ((lane % CPR) ^ kswz<CPR>(kr[it])) * 8;
      if (m > last_chunk) m = last_chunk;
      col_off[it] = m * 2;
    }
  }
  // KT: k-rows at or past kend reload row kend-1 (masked out of the MFMAs).
  template <bool KT>
  __device__ __forceinline__ void issue(int64_t k0, char* dst, int64_t kend) const {
    const unsigned lds0 = lds_base_of(dst) + wave_id() * 1024;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      int64_t k = k0 + kr[it];
      if (KT && k >= kend) k = kend - 1;
      dma_b128(base + k * ld + col_off[it], lds0 + it * WAVES * 1024);
    }
  }
  template <bool KT>
  __device__ __forceinline__ void issue_range(int64_t k0, char* dst, int64_t kend, int lo, int hi) const {
    const unsigned lds0 = lds_base_of(dst) + wave_id() * 1024;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      if (it < lo || it >= hi) continue;
      int64_t k = k0 + kr[it];
      if (KT && k >= kend) k = kend - 1;
      dma_b128(base + k * ld + col_off[it], lds0 + it * WAVES * 1024);
    }
  }
};

template <int ROWS, int NT, bool K_CONTIG, int BK>
struct OperandLoad;
template <int ROWS, int NT, int BK>
struct OperandLoad<ROWS, NT, true, BK> {
  TileLoad<ROWS, NT, BK> t;
  __device__ __forceinline__ void init(const char* b, int64_t ld, int64_t r0, int64_t n) { t.init(b, ld, r0, n); }
  template <bool KT>
  __device__ __forceinline__ void issue(int64_t k0, char* dst, int64_t kend) const {
    t.template issue<KT>(k0 * 2, dst, kend * 2);
  }
  template <bool KT>
  __device__ __forceinline__ void issue_range(int64_t k0, char* dst, int64_t kend, int lo, int hi) const {
    t.template issue_range<KT>(k0 * 2, dst, kend * 2, lo, hi);
  }
  static constexpr int ITERS = TileLoad<ROWS, NT, BK>::ITERS;
};
template <int ROWS, int NT, int BK>
struct OperandLoad<ROWS, NT, false, BK> {
  TileLoadT<ROWS, NT, BK> t;
  __device__ __forceinline__ void init(const char* b, int64_t ld, int64_t r0, int64_t n) { t.init(b, ld, r0, n); }
  template <bool KT>
  __device__ __forceinline__ void issue(int64_t k0, char* dst, int64_t kend) const {
    t.template issue<KT>(k0, dst, kend);
  }
  template <bool KT>
  __device__ __forceinline__ void issue_range(int64_t k0, char* dst, int64_t kend, int lo, int hi) const {
    t.template issue_range<KT>(k0, dst, kend, lo, hi);
  }
  static constexpr int ITERS = TileLoadT<ROWS, NT, BK>::ITERS;
};


// CNT MFMA fragments (rows r0 + 16i .. +15, k = ks*32 + 8g + 0..7) from an
// m/n-contiguous tile, two transposing reads each: within a 16-lane group,
// lane i receives element i%4 of the 4-element pieces of lanes i/4, 4+i/4,
// 8+i/4, 12+i/4, so source lane 4e+q supplies k-row (.. + e), columns
// r0+4q..+3.
template <typename T, int ROWS, int CNT>
__device__ __forceinline__ void mn_frags(const char* tile, int r0, int ks, typename Mfma<T>::frag (&f)[CNT]) {
  constexpr int ROWB = ROWS * 2;
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, src = lane & 15;
  const int k1 = ks * 32 + 8 * g + (src >> 2), k2 = k1 + 4;
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int m = r0 + i * 16 + 4 * (src & 3);
    const s16x4 a = ds_read_tr(tile + k1 * ROWB + (((m >> 3) ^ kswz<ROWS / 8>(k1)) << 4) + ((m & 7) << 1));
    const s16x4 b = ds_read_tr(tile + k2 * ROWB + (((m >> 3) ^ kswz<ROWS / 8>(k2)) << 4) + ((m & 7) << 1));
    f[i] = join_frag<typename Mfma<T>::frag>(a, b);
  }
}

// Zero the fragment slots whose k index (kbase + slot) is >= kend.
template <typename F>
__device__ __forceinline__ void mask_k(F& f, int64_t kbase, int64_t kend) {
  short* fs = (short*)&f;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (kbase + e >= kend) fs[e] = 0;
}

// Block configurations.
template <int CFG>
struct TileCfg;
template <>
struct TileCfg<0> {  // C128
  static constexpr int BM = 128, BN = 128, BK = 64, WGM = 2, WGN = 2, STAGES = 2, MIN_BLOCKS = 2;
};
template <>
struct TileCfg<1> {  // C256
  static constexpr int BM = 256, BN = 256, BK = 64, WGM = 2, WGN = 4, STAGES = 2, MIN_BLOCKS = 1;
};
template <>
struct TileCfg<2> {  // C192: 128x192, waves of 64x96, 40 KB per stage (k-contiguous B only)
  static constexpr int BM = 128, BN = 192, BK = 64, WGM = 2, WGN = 2, STAGES = 2, MIN_BLOCKS = 2;
};
// C256W: the same tile by four waves of 128x128, one on each SIMD, for long K.
// What bounds C256's loop is LDS: its waves of 128x64 read 192 KB a stage (1536
// cycles) and the loads write 64 KB (512), as long as the MFMAs (2048); these
// read 128 KB.  Five slots of 32 KB (160 KB).
template <>
struct TileCfg<3> {
  static constexpr int BM = 256, BN = 256, BK = 64, WGM = 2, WGN = 2, STAGES = 2, MIN_BLOCKS = 1;
};

// C64: 64x64, 4 waves of 32x32, four 16 KB stages, two blocks per CU: for
// outputs whose 128x128 tiles leave CUs idle.  There a k-step takes the
// latency of its loads and not its MFMA time, so more and smaller blocks with
// three stages in flight shorten it.
template <>
struct TileCfg<4> {
  static constexpr int BM = 64, BN = 64, BK = 64, WGM = 2, WGN = 2, STAGES = 4, MIN_BLOCKS = 2;
};

// s_waitcnt immediate for vmcnt(n), other counters not waited on.
constexpr int vmcnt_imm(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }

// Wait until only the loads of the stages after this one are outstanding:
// `later` of them (at most LATER) have been issued.
template <int LATER, int PER_STAGE>
__device__ __forceinline__ void wait_stage(int64_t later) {
  if (LATER == 0 || later >= LATER) __builtin_amdgcn_s_waitcnt(vmcnt_imm(LATER * PER_STAGE));
  else if constexpr (LATER > 0) wait_stage<LATER - 1, PER_STAGE>(later);
}

// C += a wave's accumulators plus the preloaded bias, element by element (C
// points at the wave tile's first element).  Offsets inside the tile are
// 32-bit (the host checks the row stride).
template <typename CT, int TM, int TN>
__device__ __forceinline__ void add_tile(CT* __restrict__ C, int c_rs, const f32x4 (&acc)[TM][TN],
                                         const float (&bias)[TN], int rows_left, int cols_left, int lr, int lg) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = i * 16 + lg * 4 + e;
      if (r >= rows_left) continue;
      CT* row = C + r * c_rs;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int c = j * 16 + lr;
        if (c < cols_left) row[c] = (CT)(acc[i][j][e] + bias[j] + (float)row[c]);
      }
    }
}

constexpr int kSlabPad = 4;  // floats between the rows of a store slab

// Full wave tiles without beta: the accumulators go through a per-wave LDS
// slab 16 rows at a time (one MFMA row of tiles, f32, rows padded by 4
// floats) and leave as row-contiguous 16-byte stores: 8 bf16/f16 or 4 f32
// per lane instead of one element per store.  The slab holds 16 x (WN + 4)
// floats; `lane` is the wave lane.  Requires 16-byte aligned rows of C.
// NT: non-temporal stores, for outputs no kernel reads soon enough to find
// them in a cache (split-K partials, summed right after, keep normal
// stores); a training step ran 0.2 ms faster with them.
template <typename CT, typename T, bool ROUND, bool NT, int TM, int TN>
__device__ __forceinline__ void store_tile_lds(CT* __restrict__ C, int c_rs, const f32x4 (&acc)[TM][TN],
                                               const float (&bias)[TN], float* slab, int lr, int lg, int lane) {
  // slab row stride in floats: 4 * LD = 16 (mod 64) puts the four 16-lane
  // groups of a store (rows lg*4 + e) on disjoint banks
  constexpr int WN = TN * 16, LD = WN + kSlabPad;
  constexpr int E = 16 / sizeof(CT);             // elements per 16-byte store
  constexpr int CHUNKS = 16 * WN / E;            // 16-byte chunks per 16-row slab
  static_assert(WN % E == 0 && CHUNKS % 64 == 0, "slab shape");
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + bias[j];
        if (ROUND) v = (float)(T)v;
        slab[(lg * 4 + e) * LD + j * 16 + lr] = v;
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int it = 0; it < CHUNKS / 64; ++it) {
      const int ch = it * 64 + lane, r = ch / (WN / E), c = (ch % (WN / E)) * E;
      const float* src = slab + r * LD + c;
      struct alignas(16) Out { CT v[E]; } out;
#pragma unroll
      for (int e = 0; e < E; ++e) out.v[e] = (CT)src[e];
      if constexpr (NT)
        __builtin_nontemporal_store(__builtin_bit_cast(f32x4, out), (f32x4*)(C + (i * 16 + r) * c_rs + c));
      else
        *(Out*)(C + (i * 16 + r) * c_rs + c) = out;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// The same through the slab for partial tiles and for rows of C that are not
// 16-byte aligned, whose 16-byte stores the hardware splits: still far fewer
// instructions than storing element by element (logits of 50257 columns,
// 16384 x 768: 1463 -> 1402 us; splitting each row at its 16-byte boundary
// instead took 1544; 1000 x 3072 at K = 768, which ended with the last row of
// tiles: 16.7 -> 13.1).  Columns past the last whole 16 bytes leave one by
// one.  Cached stores, so that the lines that two waves share are merged.
template <typename CT, typename T, bool ROUND, int TM, int TN>
__device__ __forceinline__ void store_tile_edge(CT* __restrict__ C, int c_rs, const f32x4 (&acc)[TM][TN],
                                                const float (&bias)[TN], float* slab, int rows_left, int cols_left,
                                                int lr, int lg, int lane) {
  constexpr int WN = TN * 16, LD = WN + kSlabPad;
  constexpr int E = 16 / sizeof(CT);
  const int cols = min(cols_left, WN);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i * 16 >= rows_left) break;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + bias[j];
        if (ROUND) v = (float)(T)v;
        slab[(lg * 4 + e) * LD + j * 16 + lr] = v;
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int it = 0; it < 16 * (WN / E) / 64; ++it) {
      const int ch = it * 64 + lane, r = ch / (WN / E), c = (ch % (WN / E)) * E;
      if (i * 16 + r >= rows_left || c + E > cols) continue;
      const float* src = slab + r * LD + c;
      struct Out { CT v[E]; } out;  // aligned as its elements are
#pragma unroll
      for (int e = 0; e < E; ++e) out.v[e] = (CT)src[e];
      *(Out*)(C + (i * 16 + r) * c_rs + c) = out;
    }
    if (cols % E != 0)
#pragma unroll
      for (int it = 0; it < 16 * E / 64; ++it) {
        const int q = it * 64 + lane, r = q / E, c = cols / E * E + q % E;
        if (i * 16 + r < rows_left && c < cols) C[(i * 16 + r) * c_rs + c] = (CT)slab[r * LD + c];
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// One fragment: rows r0 .. r0 + 15, k substep ks of a stage's tile of ROWS rows.
template <typename T, int ROWS, bool K_CONTIG>
__device__ __forceinline__ typename Mfma<T>::frag read_frag(const char* tile, int r0, int ks) {
  typedef typename Mfma<T>::frag frag;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  if constexpr (K_CONTIG) {
    return *(const frag*)(tile + (r0 + lr) * 128 + ((ks * 4 + lg) ^ rswz(lr)) * 16);
  } else {
    frag f[1];
    mn_frags<T, ROWS, 1>(tile, r0, ks, f);
    return f[0];
  }
}

// c += a b on accumulators that stay where they are: given the builtin, the
// compiler moves 256 of them about between the MFMAs of a loop.  It does not see
// that c is an MFMA's result, which other instructions may read only 10 states
// later: nothing may read or copy an accumulator before the s_nops that end
// wide_loop.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void mma_acc(f32x4& c, const Mfma<bf16>::frag& a, const Mfma<bf16>::frag& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+a"(c) : "v"(__builtin_bit_cast(i32x4, a)), "v"(__builtin_bit_cast(i32x4, b)));
}
__device__ __forceinline__ void mma_acc(f32x4& c, const Mfma<f16>::frag& a, const Mfma<f16>::frag& b) {
  asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
               : "+a"(c) : "v"(__builtin_bit_cast(i32x4, a)), "v"(__builtin_bit_cast(i32x4, b)));
}

// C256W's k loop.  A wave has its SIMD to itself, so nothing hides what it
// waits for but its own MFMAs: each 32-k substep's fragments are read during
// the substep before, and the loads of a stage are issued over both substeps
// of the stage two before it, A's into the slot that the ring has free, B's
// into the one that A leaves at the barrier between them.  In one burst after
// that barrier, with four slots, they stalled the wave (8192^3 1112 us; 868).
// Two or one loads a row took as long in the forward and 7% longer with
// transposed operands.
// Against C256 (us): 8192^3 917 -> 869, dX 1074 -> 927, dW 1110 -> 994; 50257
// columns dX 16384 rows 1468 -> 1268 (C192 1386), dW 1275 -> 1160; 16384 x
// 4096 at K = 4096 471 -> 461; but at K = 768 83 -> 86 and 74 -> 79 (the only wave
// of a SIMD zeroes 256 accumulators and ends with 64 s_nops; what share of that
// they have is not measured).
template <typename T, typename C, bool KT, bool A_K, bool B_K, typename LA, typename LB, int TM, int TN>
__device__ __forceinline__ void wide_loop(const LA& la, const LB& lb, f32x4 (&acc)[TM][TN], char* lds, int64_t kbeg,
                                          int64_t kend, int wm, int wn) {
  typedef typename Mfma<T>::frag frag;
  constexpr int A_BYTES = C::BM * C::BK * 2, STAGE = A_BYTES + C::BN * C::BK * 2, BK = C::BK;
  constexpr int NA = LA::ITERS, NQ = NA + LB::ITERS, R = TM + TN;
  constexpr int LPR = 4;  // loads per row of MFMAs: A's in the first substep's first rows, B's in the second's
  struct Frags { frag a[TM], b[TN]; } f0, f1;
  auto read = [&](Frags& f, const char* ta, const char* tb, int ks, int lo, int hi) {  // B's first: every row of MFMAs takes them all
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (q < lo || q >= hi) continue;
      if (q < TN) f.b[q] = read_frag<T, C::BN, B_K>(tb, wn * TN * 16 + q * 16, ks);
      else f.a[q - TN] = read_frag<T, C::BM, A_K>(ta, wm * TM * 16 + (q - TN) * 16, ks);
    }
  };
  auto mask = [&](frag& f, int64_t kfrag) {
    mask_k(f, kfrag, kend);
    asm volatile("s_nop 3" : "+v"(f));  // an MFMA may read it 2 states later
  };
  auto mask_all = [&](Frags& f, int64_t kfrag) {
#pragma unroll
    for (int j = 0; j < TN; ++j) mask(f.b[j], kfrag);
#pragma unroll
    for (int i = 0; i < TM; ++i) mask(f.a[i], kfrag);
  };
  if (kbeg >= kend) return;
  // stage 0 is in flight
  if (kbeg + BK < kend) {
    la.template issue<KT>(kbeg + BK, lds + STAGE, kend);
    lb.template issue<KT>(kbeg + BK, lds + STAGE + A_BYTES, kend);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(NQ));
  } else {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  }
  __syncthreads();
  read(f0, lds, lds + A_BYTES, 0, 0, R);
  const int lg = (threadIdx.x & 63) >> 4;
  // slots of 32 KB in a ring of five: A of stage s in slot 2 s % 5, B in the next
  char *sa = lds, *sb = lds + A_BYTES;
  auto next = [&](char* s, int n) {  // n slots on
    s += n * A_BYTES;
    return s >= lds + 5 * A_BYTES ? s - 5 * A_BYTES : s;
  };
  auto step = [&](int64_t k0, auto tail_c, auto more_c) {
    constexpr bool tail = decltype(tail_c)::value, more = decltype(more_c)::value;
    char *const na = next(sa, 2), *const nb = next(sb, 2), *const fre = next(sa, 4);
    if (tail) mask_all(f0, k0 + lg * 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (more) la.template issue_range<KT>(k0 + 2 * BK, fre, kend, i * LPR, (i + 1) * LPR);
      read(f1, sa, sb, 1, i * R / (TM - 2), (i + 1) * R / (TM - 2));
      if (i == TM - 1) {
        // all of this stage is in registers and the next one has landed
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(more ? NA : 0));
        __syncthreads();
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) mma_acc(acc[i][j], f0.a[i], f0.b[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (tail) mask_all(f1, k0 + 32 + lg * 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (more) lb.template issue_range<KT>(k0 + 2 * BK, sa, kend, i * LPR, (i + 1) * LPR);
      read(f0, na, nb, 0, i * R / (TM - 1), (i + 1) * R / (TM - 1));  // past the last stage: not used
#pragma unroll
      for (int j = 0; j < TN; ++j) mma_acc(acc[i][j], f1.a[i], f1.b[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    sa = na;
    sb = nb;
  };
  int64_t k0 = kbeg;
  for (; k0 + 2 * BK < kend; k0 += BK) step(k0, std::false_type{}, std::true_type{});
  for (; KT ? k0 + BK <= kend : k0 < kend; k0 += BK) step(k0, std::false_type{}, std::false_type{});
  if (KT && k0 < kend) step(k0, std::true_type{}, std::false_type{});
  // an MFMA's results may be read 10 states after it
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("s_nop 15" : "+a"(acc[i][j]));
}

// RS: also sum A's rows over k, from the fragments the MFMAs consume, with
// one extra MFMA against a fragment of ones (every column of its 16x16
// result is the row sum).  With split K the 32-k substeps are dealt round
// robin over the tiles_n * WGN waves that hold the same rows (one substep in
// that many per wave), each writing its own partial slot; without split K
// the waves of the first wave column of the first column tile do it all.
template <typename T, int CFG, bool A_K, bool B_K, bool KT, bool RS>
__global__ void __launch_bounds__(64 * TileCfg<CFG>::WGM * TileCfg<CFG>::WGN, TileCfg<CFG>::MIN_BLOCKS)
    gemm_tile(GemmArgs g) {
  typedef typename Mfma<T>::frag frag;
  typedef TileCfg<CFG> C;
  constexpr int BM = C::BM, BN = C::BN;
  constexpr int NT = 64 * C::WGM * C::WGN;
  constexpr int WM = BM / C::WGM, WN = BN / C::WGN;
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int BK = C::BK, ROWB = BK * 2;  // k per stage, bytes of a k-contiguous row
  constexpr int A_BYTES = BM * ROWB, STAGE = A_BYTES + BN * ROWB, S = C::STAGES;
  char* const lds = gemm_smem;

  // XCD-aware order over the whole grid: the hardware deals workgroups to
  // the 8 XCDs round-robin in dispatch order (x fastest, then y), so XCD
  // L % 8 gets every 8th block.  Each XCD is given one contiguous run of the
  // (split, batch)-major tile list instead: its blocks share A/B panels and,
  // with split K, one or two K ranges, so each L2 fetches about 1/8 of the
  // operands (dealing a plane's tiles over all XCDs made every L2 fetch
  // every split's panels).  A bijection for any grid size.
  const uint32_t nt = gridDim.x;
  uint32_t L = blockIdx.x + nt * blockIdx.y;
  {
    const uint32_t total = nt * gridDim.y, xcd = L & 7, q = total >> 3, r = total & 7;
    L = xcd * q + min(xcd, r) + (L >> 3);
  }
  const uint32_t plane = L / nt, t = L - plane * nt;
  uint32_t tm, tn;
  if (g.group > 1) {
    // `group` tile rows at a time, column by column: an XCD's blocks share B's
    // panels across the group's rows while the rows of A stay in its L2
    const uint32_t per = (uint32_t)g.group * (uint32_t)g.tiles_n, first = t / per * (uint32_t)g.group;
    const uint32_t r = t % per, rows = min((uint32_t)g.group, nt / (uint32_t)g.tiles_n - first);
    tn = r / rows, tm = first + (r - tn * rows);
  } else {
    tm = t / (uint32_t)g.tiles_n, tn = t - tm * (uint32_t)g.tiles_n;
  }
  const uint32_t split = plane / (uint32_t)g.batch, bidx = plane - split * (uint32_t)g.batch;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  int64_t kbeg = 0, kend = g.k;
  if (g.part) {
    kbeg = (int64_t)split * g.kchunk;
    kend = min(g.k, kbeg + g.kchunk);
  }

  const char* A = (const char*)g.a + (int64_t)bidx * g.a_bs * (int64_t)sizeof(T);
  const char* B = (const char*)g.b + (int64_t)bidx * g.b_bs * (int64_t)sizeof(T);
  // A_K: bytes between rows; else bytes between k-rows.  Same for B.
  const int64_t a_ldb = (A_K ? g.a_rs : g.a_cs) * (int64_t)sizeof(T);
  const int64_t b_ldb = (B_K ? g.b_cs : g.b_rs) * (int64_t)sizeof(T);

  const int lane = threadIdx.x & 63, wave = wave_id();  // scalar: the row-sum test branches on it
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  const int lr = lane & 15, lg = lane >> 4;

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  OperandLoad<BM, NT, A_K, BK> la;
  OperandLoad<BN, NT, B_K, BK> lb;
  constexpr int PER_STAGE = decltype(la.t)::ITERS + decltype(lb.t)::ITERS;  // DMA instructions per stage
  static_assert(S == 2 || (S - 2) * PER_STAGE < 64, "vmcnt range");
  la.init(A, a_ldb, m0, g.m);
  lb.init(B, b_ldb, n0, g.n);
  // Prologue: stages 0 .. S-2 in flight.
#pragma unroll
  for (int st = 0; st < S - 1; ++st) {
    if (kbeg + st * BK < kend) {
      la.template issue<KT>(kbeg + st * BK, lds + st * STAGE, kend);
      lb.template issue<KT>(kbeg + st * BK, lds + st * STAGE + A_BYTES, kend);
    }
  }
  // k-contiguous fragment rows (.. + lr) share the swizzle of lr
  const int sw = rswz(lr);
  const int rs_slots = g.part ? g.tiles_n * C::WGN : 1;
  const int rs_slot = g.part ? (int)tn * C::WGN + wn : 0;
  const bool rs_on = RS && (g.part || (tn == 0 && wn == 0));
  int rs_q = 0;  // this wave's substep counter modulo rs_slots
  f32x4 rsum[TM];
  frag ones;
#pragma unroll
  for (int i = 0; i < TM; ++i) rsum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (T)1.0f;

  int cur = 0;
  // One stage; TAIL: K ends inside it, so what lies past the end is masked.
  // The last stage alone is compiled with the masks: a test of them in every
  // stage, even one that is never taken, splits the MFMAs into short runs (K =
  // 50257 into 768 columns: 16384 rows 1443 -> 1422 us, 2048 rows 235 -> 211).
  auto step = [&](int64_t k0, auto tail_c) {
    constexpr bool tail = decltype(tail_c)::value;
    // This step's tiles have landed when at most the later stages' loads
    // (S-2 stages, if issued) are still outstanding.
    wait_stage<S - 2, PER_STAGE>((kend - 1 - k0) / BK);
    __syncthreads();
    // the next stage goes to the slot read in the previous step (every wave
    // is past it); its loads are issued after this step's first B fragment
    // reads, so the first MFMAs do not wait behind the load issue (training
    // step 22.22 -> 22.03 ms, three runs each on one box; issuing them after
    // the reads only for k-contiguous A gave nothing).  The 256x256 tiles
    // (eight MFMA rows per wave) spread the load instructions over the MFMA
    // rows of the first 32-k substep instead, so the load issue no longer
    // stalls the wave in one burst: the forward fc and lm_head launches run
    // 3.4-5.8% faster in the training step (kernel trace, two boxes); the
    // same spread lost 2-6% on the 128x128 and 128x192 tiles, which keep the
    // single burst.
    const bool more = k0 + (S - 1) * BK < kend;
    char* const nxt = lds + (cur == 0 ? S - 1 : cur - 1) * STAGE;
    const char* at = lds + cur * STAGE;
    const char* bt = at + A_BYTES;
    if constexpr (CFG == 4) {
      // A wave has its SIMD nearly to itself and few MFMAs a step, so a step
      // is as long as its chain of latencies: every fragment is read before
      // the loads are issued and the first MFMA waits, one LDS latency a step
      // instead of four.
      frag af[BK / 32][TM], bf[BK / 32][TN];
#pragma unroll
      for (int ks = 0; ks < BK / 32; ++ks) {
        const int coff = ((ks * 4 + lg) ^ sw) * 16;
        if constexpr (B_K) {
#pragma unroll
          for (int j = 0; j < TN; ++j) bf[ks][j] = *(const frag*)(bt + (wn * WN + j * 16 + lr) * ROWB + coff);
        } else {
          mn_frags<T, BN, TN>(bt, wn * WN, ks, bf[ks]);
        }
        if constexpr (A_K) {
#pragma unroll
          for (int i = 0; i < TM; ++i) af[ks][i] = *(const frag*)(at + (wm * WM + i * 16 + lr) * ROWB + coff);
        } else {
          mn_frags<T, BM, TM>(at, wm * WM, ks, af[ks]);
        }
      }
      if (more) {
        la.template issue<KT>(k0 + (S - 1) * BK, nxt, kend);
        lb.template issue<KT>(k0 + (S - 1) * BK, nxt + A_BYTES, kend);
      }
      if (tail) {
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
          const int64_t kfrag = k0 + ks * 32 + lg * 8;
#pragma unroll
          for (int j = 0; j < TN; ++j) mask_k(bf[ks][j], kfrag, kend);
#pragma unroll
          for (int i = 0; i < TM; ++i) mask_k(af[ks][i], kfrag, kend);
        }
      }
#pragma unroll
      for (int ks = 0; ks < BK / 32; ++ks) {
        const bool rs_now = rs_on && rs_q == rs_slot;
        if (RS && ++rs_q == rs_slots) rs_q = 0;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if (RS && rs_now) rsum[i] = Mfma<T>::mma(af[ks][i], ones, rsum[i]);
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::mma(af[ks][i], bf[ks][j], acc[i][j]);
        }
      }
      cur = cur == S - 1 ? 0 : cur + 1;
      return;
    }
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      const bool rs_now = rs_on && rs_q == rs_slot;
      if (RS && ++rs_q == rs_slots) rs_q = 0;
      const int coff = ((ks * 4 + lg) ^ sw) * 16;
      const int64_t kfrag = k0 + ks * 32 + lg * 8;
      // an m-contiguous A's fragments are read all at once, but one at a time
      // where the row sums' accumulators leave no registers for them
      constexpr bool A_ALL = !A_K && !(RS && CFG == 1);
      frag bfr[TN], afr[A_ALL ? TM : 1];
      if constexpr (!B_K) mn_frags<T, BN, TN>(bt, wn * WN, ks, bfr);
      if constexpr (A_ALL) mn_frags<T, BM, TM>(at, wm * WM, ks, afr);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (B_K) bfr[j] = *(const frag*)(bt + (wn * WN + j * 16 + lr) * ROWB + coff);
        if (tail) mask_k(bfr[j], kfrag, kend);
      }
      if (CFG != 1 && ks == 0 && more) {
        la.template issue<KT>(k0 + (S - 1) * BK, nxt, kend);
        lb.template issue<KT>(k0 + (S - 1) * BK, nxt + A_BYTES, kend);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (CFG == 1 && ks == 0 && more) {
          // load instructions q in [lo, hi) of this stage's list (A's, then B's)
          constexpr int NA = decltype(la)::ITERS, NQ = NA + decltype(lb)::ITERS;
          const int lo = i * NQ / TM, hi = (i + 1) * NQ / TM;
          la.template issue_range<KT>(k0 + (S - 1) * BK, nxt, kend, lo, hi);
          lb.template issue_range<KT>(k0 + (S - 1) * BK, nxt + A_BYTES, kend, lo - NA, hi - NA);
        }
        frag af;
        if constexpr (A_ALL) af = afr[i];
        else if constexpr (A_K) af = *(const frag*)(at + (wm * WM + i * 16 + lr) * ROWB + coff);
        else af = read_frag<T, BM, false>(at, wm * WM + i * 16, ks);
        if (tail) mask_k(af, kfrag, kend);
        if (RS && rs_now) rsum[i] = Mfma<T>::mma(af, ones, rsum[i]);
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::mma(af, bfr[j], acc[i][j]);
      }
    }
    cur = cur == S - 1 ? 0 : cur + 1;
  };
  if constexpr (CFG == 3) {
    wide_loop<T, C, KT, A_K, B_K>(la, lb, acc, lds, kbeg, kend, wm, wn);
  } else {
    int64_t k0 = kbeg;
    for (; KT ? k0 + BK <= kend : k0 < kend; k0 += BK) step(k0, std::false_type{});
    if (KT && k0 < kend) step(k0, std::true_type{});
  }

  // every wave is past its last LDS read: the stages become store slabs
  __syncthreads();
  float* const slab = (float*)lds + wave * (16 * (WN + kSlabPad));
  const int64_t row0 = m0 + wm * WM, col0 = n0 + wn * WN;
  if (RS && rs_on && lr == 0) {
    // lane (lg, 0) holds rows 4*lg .. 4*lg+3 of each 16-row fragment
    const int64_t slot = (int64_t)split * rs_slots + rs_slot;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t r = row0 + i * 16 + lg * 4 + e;
        if (r >= g.m) continue;
        if (g.part) {
          g.rs_part[(slot * g.batch + bidx) * g.m + r] = rsum[i][e];
        } else {
          const float v = g.round_c ? round_through(rsum[i][e], g.ab_dt) : rsum[i][e];
          st_any(g.rowsum, g.rowsum_dt, (int64_t)bidx * g.m + r, v);
        }
      }
  }
  const int rows_left = (int)min(g.m - row0, (int64_t)WM), cols_left = (int)min(g.n - col0, (int64_t)WN);
  if (rows_left <= 0 || cols_left <= 0) return;
  float bias[TN];
  if (g.part) {
#pragma unroll
    for (int j = 0; j < TN; ++j) bias[j] = 0.f;
    float* P = g.part + ((int64_t)split * g.batch + bidx) * g.m * g.n + row0 * g.n + col0;
    if (rows_left == WM && cols_left == WN && (g.n & 3) == 0 && ((uintptr_t)g.part & 15) == 0)
      store_tile_lds<float, T, false, false>(P, (int)g.n, acc, bias, slab, lr, lg, lane);
    else
      store_tile_edge<float, T, false>(P, (int)g.n, acc, bias, slab, rows_left, cols_left, lr, lg, lane);
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int c = j * 16 + lr;
    bias[j] = (g.bias && c < cols_left) ? ld_any(g.bias, g.bias_dt, col0 + c) : 0.f;
  }
  const int64_t c_es = g.c_dt == MI355X_F32 ? 4 : 2;
  char* Cb = (char*)g.c + ((int64_t)bidx * g.c_bs + row0 * g.c_rs + col0) * c_es;
  const int c_rs = (int)g.c_rs;
  const bool rnd = g.round_c && g.c_dt == MI355X_F32;  // 16-bit outputs are already rounded
  const bool full = rows_left == WM && cols_left == WN && !g.beta && ((uintptr_t)g.c & 15) == 0 &&
                    (c_rs * c_es) % 16 == 0 && (g.c_bs * c_es) % 16 == 0;
  if (full) {
    if (g.c_dt == MI355X_BF16) store_tile_lds<bf16, T, false, true>((bf16*)Cb, c_rs, acc, bias, slab, lr, lg, lane);
    else if (g.c_dt == MI355X_F16) store_tile_lds<f16, T, false, true>((f16*)Cb, c_rs, acc, bias, slab, lr, lg, lane);
    else if (rnd) store_tile_lds<float, T, true, true>((float*)Cb, c_rs, acc, bias, slab, lr, lg, lane);
    else store_tile_lds<float, T, false, true>((float*)Cb, c_rs, acc, bias, slab, lr, lg, lane);
    return;
  }
  if (g.beta) {
    if (g.c_dt == MI355X_BF16) add_tile<bf16>((bf16*)Cb, c_rs, acc, bias, rows_left, cols_left, lr, lg);
    else if (g.c_dt == MI355X_F32) add_tile<float>((float*)Cb, c_rs, acc, bias, rows_left, cols_left, lr, lg);
    else add_tile<f16>((f16*)Cb, c_rs, acc, bias, rows_left, cols_left, lr, lg);
    return;
  }
#define EDGE(CT, R) store_tile_edge<CT, T, R>((CT*)Cb, c_rs, acc, bias, slab, rows_left, cols_left, lr, lg, lane)
  if (g.c_dt == MI355X_BF16) EDGE(bf16, false);
  else if (g.c_dt == MI355X_F16) EDGE(f16, false);
  else if (rnd) EDGE(float, true);
  else EDGE(float, false);
#undef EDGE
}

// Launch one kernel instantiation; the first launch of each opts it into
// more than 64 KB of dynamic LDS when it needs that.
template <typename T, int CFG, bool A_K, bool B_K, bool KT, bool RS>
int launch_kernel(const GemmArgs& g, dim3 grid, hipStream_t s) {
  typedef TileCfg<CFG> C;
  constexpr int NT = 64 * C::WGM * C::WGN;
  constexpr size_t lds = CFG == 3 ? 163840 : C::STAGES * (size_t)(C::BM + C::BN) * C::BK * 2;
  static bool attr = false;
  if (lds > 65536 && !attr) {
    if (hipFuncSetAttribute((const void*)gemm_tile<T, CFG, A_K, B_K, KT, RS>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return fail(MI355X_ELAUNCH, "mi355x_gemm: cannot reserve %zu bytes of LDS", lds);
    attr = true;
  }
  gemm_tile<T, CFG, A_K, B_K, KT, RS><<<grid, NT, lds, s>>>(g);
  return check_launch("mi355x_gemm");
}

template <typename T, int CFG, bool KT, bool RS>
int launch_layout(const GemmArgs& g, dim3 grid, hipStream_t s) {
  const bool ak = g.a_cs == 1, bk = g.b_rs == 1;
  if constexpr (CFG == 2) {  // 192-wide B tiles are only loaded k-contiguous
    if (!bk) return fail(MI355X_EINVAL, "mi355x_gemm: 128x192 tiles need a k-contiguous B");
    if (ak) return launch_kernel<T, CFG, true, true, KT, RS>(g, grid, s);
    return launch_kernel<T, CFG, false, true, KT, RS>(g, grid, s);
  } else {
    if (ak && bk) return launch_kernel<T, CFG, true, true, KT, RS>(g, grid, s);
    if (ak) return launch_kernel<T, CFG, true, false, KT, RS>(g, grid, s);
    if (bk) return launch_kernel<T, CFG, false, true, KT, RS>(g, grid, s);
    return launch_kernel<T, CFG, false, false, KT, RS>(g, grid, s);
  }
}

template <typename T, int CFG, bool KT>
int launch_tile(GemmArgs g, int64_t batch, int splits, hipStream_t s) {
  typedef TileCfg<CFG> C;
  const int tm = (int)ceil_div(g.m, C::BM), tn = (int)ceil_div(g.n, C::BN);
  g.tiles_n = tn;
  g.batch = (int)batch;
  // Row by row reads all of B for each tile row: when B is past two of an
  // XCD's 4 MB L2, walk as many tile rows together as keep their part of A in
  // half of it (logits of 50257 columns at K = 768: 2048 rows 230 -> 161 us, 8192
  // rows 799 -> 764 us, 16384 rows the same).  From one L2 on where that is all
  // of A: then each XCD reads its part of B once (512 x 4096 at K = 1024 13.1 ->
  // 9.5 us and with an n-contiguous B 15.9 -> 9.5, 1021 x 3072 at K = 768 13.0 ->
  // 11.2; with more of A 2048 x 768 at K = 3072 19.6 -> 21.0; two tile rows gain
  // nothing, 65 x 4096 at K = 640 5.4 -> 5.6).
  // Not where a short K leaves the stores of C in front, past the 256 MB
  // Infinity Cache: in rows that are not 16-byte aligned, whose lines are written
  // in parts, which row by row meet in the L2 sooner (16384 x 30001 at K = 256 /
  // 512 / 640 / 704, us: in groups 539 / 658 / 699 / 691, row by row 374 / 561 / 653
  // / 698; 4096 x 30001 at K = 512 146 / 154); and in one group (5644 x 50257 at K =
  // 64 295, row by row 268).
  g.group = 1;
  const int64_t k = min(g.k, g.kchunk), b_bytes = g.n * k * (int64_t)sizeof(T);
  const int64_t c_es = g.c_dt == MI355X_F32 ? 4 : 2, rows = (2 << 20) / (C::BM * k * (int64_t)sizeof(T));
  const bool c_far = !g.part && g.m * g.n * c_es > (256 << 20);
  const bool c_parts = (g.c_rs * c_es % 16 != 0 || (uintptr_t)g.c % 16 != 0) && c_far && k < 704;
  if (!c_parts && (b_bytes > (8 << 20) || (b_bytes > (4 << 20) && !c_far && tm > 2 && tm <= rows)))
    g.group = (int)(rows < 1 ? 1 : rows > tm ? tm : rows);
  dim3 grid((unsigned)(tm * tn), (unsigned)(batch * splits));
  if constexpr (CFG != 3) {  // which has no row sums
    if (g.rowsum) return launch_layout<T, CFG, KT, true>(g, grid, s);
  }
  return launch_layout<T, CFG, KT, false>(g, grid, s);
}

}  // namespace

template <typename T, bool KT>
int gemm_tiles(const GemmArgs& g, int64_t batch, int cfg, int splits, hipStream_t s) {
  switch (cfg) {
    case 1: return launch_tile<T, 1, KT>(g, batch, splits, s);
    case 2: return launch_tile<T, 2, KT>(g, batch, splits, s);
    case 3: return launch_tile<T, 3, KT>(g, batch, splits, s);
    case 4: return launch_tile<T, 4, KT>(g, batch, splits, s);
    default: return launch_tile<T, 0, KT>(g, batch, splits, s);
  }
}

}  // namespace mi
