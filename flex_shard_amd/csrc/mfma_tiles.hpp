// Shared pieces of the MFMA tile kernels (bf16 Newton-Schulz GEMM, FP8
// blockwise GEMM): launch parameters, the XCD-aware workgroup -> tile order,
// the LDS-staged epilogue, and the global->LDS load helpers.
#pragma once
#include "common.hpp"

#include <atomic>
#include <cmath>
#include <type_traits>

namespace fsh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct GemmParams {
  const uint16_t* A;
  const uint16_t* B;
  const uint16_t* D;
  uint16_t* C;
  uint16_t* Ct;
  int64_t M, N, K;
  int64_t lda, ldb, ldd, ldc, ldct;
  int64_t sA, sB, sD, sC, sCt;
  float alpha, beta;
  float diag_add;         // added to C[i][i] before the rounding
  int32_t tiles_m, tiles_n;
  // Not 0: the product is symmetric.  Tile rows are `symmetric` tile columns high; only the tiles from a tile row's
  // diagonal on are computed, those right of the diagonal's tile row are mirrored.
  int32_t symmetric;
  int32_t k_major;        // A is [K, M] and B is [K, N]: the product is A^T B (large-tile kernel only)
  int32_t tiles_per_matrix;
  int64_t work_items;     // tiles_per_matrix * batch
  int64_t items_per_xcd;  // ceil(work_items / 8); the grid has 8 * items_per_xcd workgroups
  // Muon update fused into the epilogue (large-tile kernel only).  When
  // update_ptrs is not null, C and D are ignored: matrix b of the batch is the
  // separately allocated parameter at update_ptrs[b] (row stride ldc), and the
  // epilogue stores  p = bf16(bf16(p * decay) + neg_lr * d),  d = bf16(acc)
  // (d scaled by dir_scale and rounded first when that is not 1): the
  // product itself is never written.
  const int64_t* update_ptrs;
  float update_decay, update_neg_lr, update_dir_scale;
#ifdef FSH_TRACE
  uint64_t* trace;
#endif
};
#ifdef FSH_TRACE
#define FSH_STAMP(slot) do { if (p.trace && threadIdx.x == 0) p.trace[blockIdx.x * 16 + (slot)] = __builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define FSH_STAMP(slot) do {} while (0)
#endif

// Several problems served by one launch: problem i
// owns the workgroup ids [first_workgroup[i], first_workgroup[i+1]), each run
// a multiple of 8 long so that the id -> XCD mapping is the same for all.
// Workgroups are dispatched in id order, so the host lists the problem with
// the longest tiles first and the short ones fill the tail of the long ones.
template <int N>
struct GemmLaunchOf {
  static constexpr int kMaxProblems = N;
  GemmParams problem[N];
  int32_t first_workgroup[N];  // INT32_MAX past the last problem
  int32_t total_workgroups;
};
using GemmLaunch = GemmLaunchOf<4>;  // the large-tile kernel (a longer lookup costs its resident form scalar registers)

constexpr int kXcds = 8;         // accelerator dies, each with its own L2
constexpr int kGroupTilesM = 4;  // tile rows walked together

// Tile t of a (non-symmetric) matrix in the patch order described below.
__device__ inline void tile_in_order(const GemmParams& p, int t, int* tm, int* tn, int rows_together = kGroupTilesM) {
  const int group_span = rows_together * p.tiles_n;
  const int first_m = (t / group_span) * rows_together;
  const int rows = min(p.tiles_m - first_m, rows_together);
  const int within = t % group_span;
  *tm = first_m + within % rows;
  *tn = within / rows;
}

// Workgroup id -> (batch, tile row, tile column).  Workgroups are handed to
// the 8 XCDs round-robin by id, and an XCD holds 32 of the large-tile
// workgroups at a time (one per CU), so XCD x is given the contiguous run
// [x, x+1) * items_per_xcd of an ordering in which 32 neighbours form a 4 x 8
// patch of tiles of one matrix: its L2 then serves 12 distinct operand panels
// per k-tile instead of 33.  Returns false for the padding ids at the end of
// an XCD's run.
__device__ inline bool tile_of_workgroup(const GemmParams& p, int64_t id, int64_t* batch, int* tm, int* tn,
                                         int rows_together = kGroupTilesM) {
  const int64_t slot = id / kXcds;
  const int64_t item = (id % kXcds) * p.items_per_xcd + slot;
  if (item >= p.work_items) return false;
  const int tiles = p.tiles_per_matrix;
  *batch = item / tiles;
  int t = static_cast<int>(item % tiles);
  if (p.symmetric) {
    // Upper triangle row by row: row r holds columns symmetric * r ..
    // tiles_n-1.  One matrix's triangle (36 tiles of a 2048^2 result) is about
    // what an XCD holds at a time, and it needs only the 8 row panels of the
    // operand.
    int r = 0;
    for (int len = p.tiles_n; t >= len; len -= p.symmetric) {
      t -= len;
      ++r;
    }
    *tm = r;
    *tn = p.symmetric * r + t;
    return true;
  }
  tile_in_order(p, t, tm, tn, rows_together);
  return true;
}

// Values that are the same in every lane but that the compiler cannot prove
// so: moved to scalar registers.
__device__ __forceinline__ int uniform_i32(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v & 0xFFFFFFFFLL)));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* ptr) {
  return reinterpret_cast<T*>(uniform_i64(reinterpret_cast<int64_t>(ptr)));
}

// Stores a [rows][row_bytes] bf16 image held in LDS (pitch bytes apart) to
// global rows `ld` elements apart, 16 bytes per lane, cut at rows_left x
// cols_left (a multiple of 8).  `dst` is the same in every lane: each store is
// a scalar base (advanced per pass) plus one 32-bit lane offset, so the passes
// share a single address register.
template <int kRows, int kRowBytes, int kPitch>
__device__ inline void store_staged_rows(const uint8_t* region, uint16_t* dst, int64_t ld, int rows_left, int cols_left, int lane) {
  constexpr int kLanesPerRow = kRowBytes / 16;
  constexpr int kRowsPerPass = 64 / kLanesPerRow;
  static_assert(kRowBytes % 16 == 0 && 64 % kLanesPerRow == 0 && kRows % kRowsPerPass == 0, "staged store shape");
  static_assert(kPitch % 16 == 0, "rows are read 16 bytes at a time");
  const int r0 = lane / kLanesPerRow, chunk = lane % kLanesPerRow;
  const uint32_t lane_off = static_cast<uint32_t>(r0) * static_cast<uint32_t>(ld * 2) + chunk * 16;
  uint8_t* base = uniform_ptr(reinterpret_cast<uint8_t*>(dst));
  const int64_t pass_bytes = uniform_i64(static_cast<int64_t>(kRowsPerPass) * ld * 2);
  const int rows = chunk * 8 < cols_left ? rows_left : 0;  // of this lane's columns
#pragma unroll
  for (int pass = 0; pass < kRows / kRowsPerPass; ++pass) {
    const int r = pass * kRowsPerPass + r0;
    const uint8_t* src = region + r * kPitch + chunk * 16;
    const u32x4 v = *reinterpret_cast<const u32x4*>(src);
    if (r < rows) *reinterpret_cast<u32x4*>(base + pass * pass_bytes + lane_off) = v;
  }
}

// Two floats -> packed bf16 pair (low half = first), round to nearest even:
// one v_cvt_pk_bf16_f32 on gfx950.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Half of a wave's D tile (its upper or lower kWaveM/2 rows), loaded the way
// C leaves: 16 bytes per lane, 256 contiguous bytes per row (in accumulator
// layout a load instruction would touch 32 rows with 16 bytes each).  Both
// halves are requested when the epilogue starts; the lower one lands while
// the upper one is being used.  (Requesting a half before the last k-tile
// was tried: with 256 accumulators live the extra 64 registers spill.)
template <typename Cfg>
struct DRows {
  static constexpr int kLanesPerRow = Cfg::kWaveN * 2 / 16, kRowsPerPass = 64 / kLanesPerRow;
  static constexpr int kPasses = Cfg::kWaveM / 2 / kRowsPerPass;
  u32x4 t[kPasses];
};

// `d` is matrix `batch` of D (row stride ldd elements).
template <typename Cfg>
__device__ __forceinline__ void load_d_rows_from(const uint16_t* d, int64_t ldd, int64_t m0, int64_t n0, int wm, int wn,
                                                 int lane, int half, int rows_left, int cols_left, DRows<Cfg>& rows) {
  using R = DRows<Cfg>;
  const int r0 = lane / R::kLanesPerRow, chunk = lane % R::kLanesPerRow;
  const uint32_t lane_off = static_cast<uint32_t>(r0) * static_cast<uint32_t>(ldd * 2) + chunk * 16;
  const uint8_t* base = uniform_ptr(reinterpret_cast<const uint8_t*>(
      d + (m0 + wm * Cfg::kWaveM + half * (Cfg::kWaveM / 2)) * ldd + n0 + wn * Cfg::kWaveN));
  const int64_t pass_bytes = uniform_i64(static_cast<int64_t>(R::kRowsPerPass) * ldd * 2);
  const int live = chunk * 8 < cols_left ? rows_left : 0;  // rows of this lane's columns
#pragma unroll
  for (int q = 0; q < R::kPasses; ++q) {
    rows.t[q] = u32x4{0, 0, 0, 0};
    if (q * R::kRowsPerPass + r0 < live) rows.t[q] = *reinterpret_cast<const u32x4*>(base + q * pass_bytes + lane_off);
  }
}

// Orders the LDS traffic of one wave: lanes exchange data through the wave's
// private staging region, which the hardware serves in program order; this
// only keeps the compiler from moving a lane's reads above other lanes'
// writes.  No counter is waited for and no workgroup barrier is taken.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Four values of one column and four consecutive rows out of a bf16 image with
// rows in LDS: within 16 lanes, lane 4 j + q passes the address of columns
// 4 q .. 4 q + 3 of row j, and lane t receives column t of rows 0 .. 3.
__device__ __forceinline__ u32x2 read_lds_transposed(const uint8_t* at) {
  typedef short i16x4 __attribute__((__vector_size__(4 * sizeof(short))));
  typedef __attribute__((address_space(3))) i16x4* lds_i16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)(const_cast<uint8_t*>(at))));
}

// Epilogue of the large-tile kernel, staged through LDS.
//
// The accumulate is issued as mfma(B, A), so accumulator r of block (i, j)
// belongs to output row m = lane%16 and column n = 4*(lane/16) + r of the
// 16x16 block.  In that layout a store instruction would touch 16 rows with
// 32 bytes each, and the transposed output would leave as 2-byte stores.
// Instead:
//   1. D is loaded row-wise (16 bytes per lane) into the staging region; the
//      finals = bf16(fma(beta, D, alpha*acc)) are computed in registers and
//      written to LDS as [row][col], each over the D value it used;
//   2. the wave reads its region back row-wise and stores C as 16 bytes per
//      lane, 256 contiguous bytes per row;
//   3. a transposed (or mirrored) output is read across the image: lane t of
//      group g of 16 takes column t of 16, rows 8 g .. 8 g + 7 of 32, in two
//      transposing reads, and 64 contiguous bytes of 16 output rows leave per store.
// The LDS row pitch is the row plus 16 bytes: 8-byte writes of 32 lanes (16
// rows, two groups of columns) then cover all banks, and rows are read 16 bytes
// at a time.
//
// The upper and then the lower 64 rows of the wave's 128x128 sub-tile are
// taken in turn, in a staging region of 17 KB per wave that only the wave
// itself touches.  The region then fits beside two of the k loop's operand
// slots, which receive the next tile's first operands while this runs, and no
// step needs a workgroup barrier (whose memory fence would wait
// for those loads).
template <typename Cfg>
struct HalfTileEpilogue {
  static constexpr int kRows = Cfg::kWaveM / 2;                 // 64
  static constexpr int kPitch = Cfg::kWaveN * 2 + 16;           // [row][col] image
  static constexpr int kRegion = kRows * kPitch;
  static constexpr int kLdsBytes = Cfg::WM * Cfg::WN * kRegion;
};

// kMode fixes the flags that every final depends on, so that the 256 finals
// of a lane are straight-line code (with the flags read at run time the
// compiler keeps a branch per group of four finals, and the waits at every
// join serialize the epilogue):
//   kEpiGeneric  any combination, flags read at run time
//   kEpiPlain    C = bf16(acc): no D, no diagonal term, alpha == 1
//   kEpiPoly     C = bf16(fma(beta, D, alpha * acc) + diag): D, alpha and the diagonal term
//   kEpiUpdate   Muon update of separately allocated parameters (see GemmParams::update_ptrs)
constexpr int kEpiGeneric = 0, kEpiPlain = 1, kEpiPoly = 2, kEpiUpdate = 3;

// (Always inlined: as a real call the accumulators and the launch's problem
// table would have to live in scratch memory.)
template <typename Cfg, int kMode, bool kRagged>
__device__ __forceinline__ void store_tile_in_halves_as(const GemmParams& p, int64_t batch, int64_t m0, int64_t n0, int wm,
                                               int wn, int lane, bool mirror, const f32x4 (&acc)[Cfg::TM][Cfg::TN],
                                               uint8_t* staging) {
  using Epi = HalfTileEpilogue<Cfg>;
  using R = DRows<Cfg>;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, HM = TM / 2;
  static_assert(TM % 2 == 0 && Epi::kRows == HM * 16, "two halves of whole 16-row blocks");
  const bool has_d = kMode == kEpiPlain ? false : (kMode == kEpiPoly || kMode == kEpiUpdate) ? true : p.D != nullptr;
  // (a pointer loaded from a table is a per-lane value to the compiler: said to be uniform here)
  uint16_t* C = kMode == kEpiUpdate ? reinterpret_cast<uint16_t*>(uniform_i64(p.update_ptrs[batch])) : p.C + batch * p.sC;
  const uint16_t* D = kMode == kEpiUpdate ? C : p.D + batch * p.sD;
  const int64_t ldd = kMode == kEpiUpdate ? p.ldc : p.ldd;
  // A symmetric product mirrors its off-diagonal tiles into the lower triangle.
  uint16_t* Ct = mirror ? C : (p.Ct ? p.Ct + batch * p.sCt : nullptr);
  const int64_t ldct = mirror ? p.ldc : p.ldct;
  const int64_t wave_row = m0 + wm * Cfg::kWaveM, wave_col = n0 + wn * Cfg::kWaveN;
  // Rows and columns of the wave's sub-tile that exist (0 or less: none).
  const auto left = [](int64_t size, int64_t at) { return kRagged && size - at < 256 ? static_cast<int>(size - at) : 256; };
  const int rows_left = left(p.M, wave_row), cols_left = left(p.N, wave_col);
  uint8_t* region = staging + (wm * Cfg::WN + wn) * Epi::kRegion;
  const int r_lane = lane & 15, c_lane = 4 * (lane >> 4);
  const bool unit_alpha = (kMode == kEpiPlain || kMode == kEpiUpdate) ? true : kMode == kEpiPoly ? false : p.alpha == 1.0f;
  // Block tiles and wave sub-tiles are square, so C's diagonal runs through
  // the (i, i) blocks of the diagonal sub-tiles of the diagonal tiles.
  const bool on_diagonal = kMode != kEpiPlain && kMode != kEpiUpdate && p.diag_add != 0.0f && m0 == n0 && wm == wn;

  // The lower half of D is requested once the upper half has left its
  // registers for LDS, and lands while the upper half is worked on.
  DRows<Cfg> drows[2];
  if (has_d) load_d_rows_from<Cfg>(D, ldd, m0, n0, wm, wn, lane, 0, rows_left, cols_left, drows[0]);
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    if (has_d) {
      // stage_d_rows with the half's rows at the top of the region
      const int r0 = lane / R::kLanesPerRow, chunk = lane % R::kLanesPerRow;
#pragma unroll
      for (int q = 0; q < R::kPasses; ++q) {
        uint8_t* d = region + (r0 + q * R::kRowsPerPass) * Epi::kPitch + chunk * 16;
        *reinterpret_cast<u32x4*>(d) = drows[hf].t[q];
      }
      if (hf == 0) load_d_rows_from<Cfg>(D, ldd, m0, n0, wm, wn, lane, 1, rows_left - Epi::kRows, cols_left, drows[1]);
      wave_lds_sync();
    }
#pragma unroll
    for (int ih = 0; ih < HM; ++ih) {
      u32x2 fin[TN];  // packed bf16 finals of this 16-row block, accumulator layout
      const int i = hf * HM + ih;
      u32x2 dv[TN];
      if (has_d) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          dv[j] = *reinterpret_cast<const u32x2*>(region + (ih * 16 + r_lane) * Epi::kPitch + (j * 16 + c_lane) * 2);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = unit_alpha ? acc[i][j][t] : p.alpha * acc[i][j][t];
        if (kMode == kEpiUpdate) {
          // The rounding sequence of the separate update kernel: direction
          // to bf16 (scaled and rounded again when the scale is not 1),
          // decayed parameter to bf16, then one multiply and one add.
          const uint32_t d01 = pack_bf16x2(v[0], v[1]), d23 = pack_bf16x2(v[2], v[3]);
          float d[4] = {u32_as_f32(d01 << 16), u32_as_f32(d01 & 0xFFFF0000u), u32_as_f32(d23 << 16),
                        u32_as_f32(d23 & 0xFFFF0000u)};
          if (p.update_dir_scale != 1.0f) {
            const uint32_t s01 = pack_bf16x2(d[0] * p.update_dir_scale, d[1] * p.update_dir_scale);
            const uint32_t s23 = pack_bf16x2(d[2] * p.update_dir_scale, d[3] * p.update_dir_scale);
            d[0] = u32_as_f32(s01 << 16); d[1] = u32_as_f32(s01 & 0xFFFF0000u);
            d[2] = u32_as_f32(s23 << 16); d[3] = u32_as_f32(s23 & 0xFFFF0000u);
          }
          const uint32_t p01 = pack_bf16x2(u32_as_f32(dv[j].x << 16) * p.update_decay,
                                           u32_as_f32(dv[j].x & 0xFFFF0000u) * p.update_decay);
          const uint32_t p23 = pack_bf16x2(u32_as_f32(dv[j].y << 16) * p.update_decay,
                                           u32_as_f32(dv[j].y & 0xFFFF0000u) * p.update_decay);
          v[0] = u32_as_f32(p01 << 16) + p.update_neg_lr * d[0];
          v[1] = u32_as_f32(p01 & 0xFFFF0000u) + p.update_neg_lr * d[1];
          v[2] = u32_as_f32(p23 << 16) + p.update_neg_lr * d[2];
          v[3] = u32_as_f32(p23 & 0xFFFF0000u) + p.update_neg_lr * d[3];
        } else if (has_d) {
          v[0] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].x << 16), v[0]);
          v[1] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].x & 0xFFFF0000u), v[1]);
          v[2] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].y << 16), v[2]);
          v[3] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].y & 0xFFFF0000u), v[3]);
        }
        if (kMode != kEpiPlain && kMode != kEpiUpdate && i == j) {
          // a select per final rather than a branch per block (adding zero
          // elsewhere would turn a -0 into +0)
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = (on_diagonal && r_lane == c_lane + t) ? v[t] + p.diag_add : v[t];
        }
        fin[j] = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
      // A lane's finals replace exactly the D values it read itself.
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *reinterpret_cast<u32x2*>(region + (ih * 16 + r_lane) * Epi::kPitch + (j * 16 + c_lane) * 2) = fin[j];
    }
    if (hf == 1) FSH_STAMP(9);
    wave_lds_sync();
    store_staged_rows<Epi::kRows, Cfg::kWaveN * 2, Epi::kPitch>(
        region, C + (wave_row + hf * Epi::kRows) * p.ldc + wave_col, p.ldc, rows_left - hf * Epi::kRows, cols_left, lane);
    if (hf == 1) FSH_STAMP(10);
    if (Ct != nullptr) {  // uniform over the workgroup
      const int t = lane & 15, g = lane >> 4;
      const int64_t lane_off = t * ldct * 2 + g * 16;
      uint8_t* base = uniform_ptr(reinterpret_cast<uint8_t*>(Ct + wave_col * ldct + wave_row + hf * Epi::kRows));
      const int64_t block_bytes = uniform_i64(32 * ldct);
      const uint8_t* from = region + (8 * g + (t >> 2)) * Epi::kPitch + (t & 3) * 8;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int rb = 0; rb < Epi::kRows / 32; ++rb) {
          const u32x2 lo = read_lds_transposed(from + rb * 32 * Epi::kPitch + j * 32);
          const u32x2 hi = read_lds_transposed(from + (rb * 32 + 4) * Epi::kPitch + j * 32);
          if (!kRagged || (j * 16 + t < cols_left && rb * 32 + 8 * g < rows_left - hf * Epi::kRows))
            *reinterpret_cast<u32x4*>(base + j * block_bytes + rb * 64 + lane_off) = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
      }
    }
    if (hf == 0) FSH_STAMP(8);
    if (hf == 0) wave_lds_sync();  // before the lower half overwrites the region
  }
}

template <typename Cfg, bool kRagged>
__device__ __forceinline__ void store_tile_in_halves(const GemmParams& p, int64_t batch, int64_t m0, int64_t n0, int wm, int wn,
                                            int lane, bool mirror, const f32x4 (&acc)[Cfg::TM][Cfg::TN],
                                            uint8_t* staging) {
  // uniform over the launch's problem, so one branch per tile
  const bool has_d = p.D != nullptr, diag = p.diag_add != 0.0f, unit_alpha = p.alpha == 1.0f;
  if (p.update_ptrs != nullptr)
    store_tile_in_halves_as<Cfg, kEpiUpdate, kRagged>(p, batch, m0, n0, wm, wn, lane, mirror, acc, staging);
  else if (!has_d && !diag && unit_alpha)
    store_tile_in_halves_as<Cfg, kEpiPlain, kRagged>(p, batch, m0, n0, wm, wn, lane, mirror, acc, staging);
  else if (has_d && !unit_alpha)
    store_tile_in_halves_as<Cfg, kEpiPoly, kRagged>(p, batch, m0, n0, wm, wn, lane, mirror, acc, staging);
  else
    store_tile_in_halves_as<Cfg, kEpiGeneric, kRagged>(p, batch, m0, n0, wm, wn, lane, mirror, acc, staging);
}

// gfx950 loads 16 bytes per lane from global memory straight into LDS: lane l
// of a wave writes LDS bytes [M0 + 16 l, M0 + 16 l + 16).  The address is a
// uniform 64-bit base plus a 32-bit per-lane offset.  Inline asm: the compiler
// neither reorders these against other memory operations nor counts them.  The
// instruction set asks for one wait state between a scalar write of M0 and a
// load to LDS, which the compiler inserts for its own instructions only.  It
// costs the large-tile products 0.5 % (48 Newton-Schulz matrices 16.28 -> 16.36 ms),
// as an idle state or as an addition to the lane's address that would be a
// scalar one otherwise.
// `lds_step`, a constant after unrolling, is added on the way into M0: the
// addresses of a k-tile's requests then need no scalar registers of their own.
__device__ __forceinline__ void dma_load_16(uint32_t voffset, const uint8_t* base, uint32_t lds_addr, uint32_t lds_step) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voffset), "s"(base), "s"(lds_addr),
               "i"(lds_step) : "memory", "scc");
}
// The same with a per-lane 64-bit address.
__device__ inline void dma_load_16_at(const uint8_t* src, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_addr) : "memory");
}
template <int kInFlight>
__device__ inline void wait_for_dma_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kInFlight) : "memory"); }
__device__ inline void wait_for_dma_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// 4 bytes per lane from a uniform base plus a 32-bit per-lane offset: lane l
// writes LDS bytes [M0 + 4 l, M0 + 4 l + 4).
__device__ inline void dma_touch_4(uint32_t voffset, const uint8_t* base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voffset), "s"(base), "s"(lds_addr) : "memory");
}

// Eight bf16 of a row that ends at column `cols`, starting at column `col`
// (< cols); 16-byte access when `vec` allows it, columns past the end as zero.
__device__ __forceinline__ u32x4 load_row_piece(const uint16_t* row, int64_t col, int64_t cols, bool vec) {
  if (vec && col + 8 <= cols) return *reinterpret_cast<const u32x4*>(row + col);
  uint32_t e[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) e[t] = col + t < cols ? row[col + t] : 0u;
  return u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
}
__device__ __forceinline__ void store_row_piece(uint16_t* row, int64_t col, int64_t cols, bool vec, u32x4 v) {
  if (vec && col + 8 <= cols) {
    *reinterpret_cast<u32x4*>(row + col) = v;
    return;
  }
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int t = 0; t < 8; ++t)
    if (col + t < cols) row[col + t] = static_cast<uint16_t>(w[t >> 1] >> (16 * (t & 1)));
}
__device__ __forceinline__ bool rows_are_16_byte(const uint16_t* p, int64_t ld) {
  return (ld & 7) == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// A wave's [kRows][kCols] image in LDS to `out` rows [row0, +) x columns
// [col0, +), cut at rows x cols, whole row segments per store instruction.
// `finish` has the last word on eight bf16 values of a lane's columns
// [column_of_lane, +8).
template <int kCols>
__device__ __forceinline__ int image_column_of_lane(int lane) {
  return lane % (kCols / 8) * 8;
}
template <int kRows, int kCols, int kPitch, typename Finish>
__device__ __forceinline__ void store_wave_image(const uint8_t* region, uint16_t* out, int64_t ld, int64_t row0,
                                                 int64_t col0, int64_t rows, int64_t cols, int lane, Finish finish) {
  constexpr int kLanesPerRow = kCols / 8, kRowsPerPass = 64 / kLanesPerRow;
  const bool vec = rows_are_16_byte(out, ld);
  const int r0 = lane / kLanesPerRow;
  const int64_t col = col0 + image_column_of_lane<kCols>(lane);
  if (col >= cols) return;
#pragma unroll
  for (int pass = 0; pass < kRows / kRowsPerPass; ++pass) {
    const int r = pass * kRowsPerPass + r0;
    if (row0 + r >= rows) break;
    const uint8_t* src = region + r * kPitch + image_column_of_lane<kCols>(lane) * 2;
    const u32x2 lo = *reinterpret_cast<const u32x2*>(src);
    const u32x2 hi = *reinterpret_cast<const u32x2*>(src + 8);
    store_row_piece(out + (row0 + r) * ld, col, cols, vec, finish(u32x4{lo.x, lo.y, hi.x, hi.y}));
  }
}
template <int kRows, int kCols, int kPitch>
__device__ __forceinline__ void store_wave_image(const uint8_t* region, uint16_t* out, int64_t ld, int64_t row0,
                                                 int64_t col0, int64_t rows, int64_t cols, int lane) {
  store_wave_image<kRows, kCols, kPitch>(region, out, ld, row0, col0, rows, cols, lane, [](const u32x4& v) { return v; });
}

// What a launch of a tile kernel takes, from measurements: tiles of the chip's
// one round at a time, per k-tile the less the emptier the round is (fewer
// workgroups share a compute unit, and with half the chip busy the clock stays
// at 2.3 instead of 1.6 GHz), and a start and end per round.
struct TileShape {
  int64_t m, n;
  double round;              // tiles the chip holds at once
  double empty, half, full;  // us per k-tile of a round that is nearly empty, half full, full
  double ends;               // us a round spends starting and ending
};
inline double rounds_us(const TileShape& shape, double tiles, double tile_ktiles, double max_ktiles) {
  const double rounds = tile_ktiles / max_ktiles / shape.round, whole = floor(rounds), part = rounds - whole;
  double per_ktile = whole * shape.full;
  if (part > 0.0)
    per_ktile += part <= 0.5 ? shape.empty + (shape.half - shape.empty) * 2.0 * part
                             : shape.half + (shape.full - shape.half) * (2.0 * part - 1.0);
  return 3.0 + per_ktile * max_ktiles + shape.ends * fmax(1.0, ceil(tiles / shape.round));
}

template <typename Kernel>
int reserve_lds(Kernel kernel, int bytes) {
  if (bytes <= 64 * 1024) return FSH_OK;
  hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (err != hipSuccess) return fail(FSH_EHIP, "gemm: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(err));
  return FSH_OK;
}


// Compute units of the current device (0 when the query fails).
inline int64_t compute_units() {
  static int cached[64] = {0};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 0;
  if (cached[device] == 0) {
    int count = 0;
    if (hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    cached[device] = count;
  }
  return cached[device];
}

// The attribute is per device and function, and sticky: it is set once per
// device and kernel, whichever host thread gets there first (setting it
// twice is harmless).
struct LdsReservation {
  std::atomic<uint64_t> devices{0};
};
template <typename Kernel>
int reserve_lds_once(LdsReservation& done, Kernel kernel, int bytes) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) device = 0;
  const uint64_t bit = (device >= 0 && device < 64) ? (1ull << device) : 0;
  if (bit && (done.devices.load(std::memory_order_acquire) & bit)) return FSH_OK;
  if (int rc = reserve_lds(kernel, bytes)) return rc;
  if (bit) done.devices.fetch_or(bit, std::memory_order_release);
  return FSH_OK;
}

}  // namespace
}  // namespace fsh
