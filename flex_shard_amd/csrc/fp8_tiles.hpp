// The scaled FP8 product, a tile at a time, and the kernel of the small tiles:
// few tokens, few columns, anything that does not fill the chip with the
// 256 x 256 tiles of fp8_linear.hip.
#pragma once
#include "mfma_tiles.hpp"

namespace fsh {
namespace {

typedef int v8i32 __attribute__((ext_vector_type(8)));

struct Fp8GemmParams {
  const uint8_t* xq;
  const float* xs;   // [k / 128][m]
  const uint8_t* wq;
  const float* ws;   // block scales: element (output-column block cb, k-block kb) at ws[cb * ws_cb + kb * ws_kb]
  const float* cs;   // per-column scales [k / 128][n] (the other kernel variant)
  uint16_t* out;
  const uint16_t* bias;  // [n] added to the rounded product, or null
  int64_t m, n, k;
  int64_t ldxq, ldwq, ldo, ws_cb, ws_kb;
  GemmParams schedule;  // tile order; its work items are the tiles computed whole
  // Workgroups [whole_grid, ...) take the remaining tiles (in the same order)
  // as two half tiles each, half_items in all (256 x 256 kernel only).
  int64_t whole_grid, half_items, half_items_per_xcd;
};

// The bias of eight output columns of a lane, added to the product's bf16
// values where they are stored: bf16(fp32(bf16(product)) + fp32(bias)), the
// bits of a separate addition of bf16 tensors without its pass over the output
// (read and write again: 7.3 us at 1000 x 5120, and a launch).
struct BiasOfLane {
  float value[8];
  __device__ __forceinline__ BiasOfLane(const uint16_t* bias, int64_t col, int64_t n) {
#pragma unroll
    for (int e = 0; e < 8; ++e) value[e] = col + e < n ? bf16_bits_to_f32(bias[col + e]) : 0.0f;
  }
  __device__ __forceinline__ u32x4 operator()(const u32x4& v) const {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = pack_bf16x2(u32_as_f32(d[j] << 16) + value[2 * j], u32_as_f32(d[j] & 0xFFFF0000u) + value[2 * j + 1]);
    return u32x4{w[0], w[1], w[2], w[3]};
  }
};

// A wave's finished image to the output, with the bias if there is one.
template <int kRows, int kCols, int kPitch>
__device__ __forceinline__ void store_fp8_product(const uint8_t* region, const Fp8GemmParams& p, int64_t row0, int64_t col0, int lane) {
  if (p.bias)
    store_wave_image<kRows, kCols, kPitch>(region, p.out, p.ldo, row0, col0, p.m, p.n, lane,
                                           BiasOfLane(p.bias, col0 + image_column_of_lane<kCols>(lane), p.n));
  else
    store_wave_image<kRows, kCols, kPitch>(region, p.out, p.ldo, row0, col0, p.m, p.n, lane);
}

// acc[r] += (product[r] * row_scale) * (column_scales of lane 4 block + r of this
// lane's row of 16; block is a constant after unrolling).  The broadcast is the
// multiply-add's own operand modifier (the compiler keeps a separate move per
// element when given the builtin).  column_scales comes from LDS, not from the
// vector ALU, so the modifier's read needs no wait states.
template <int N>
__device__ __forceinline__ float fold_one_with_row_broadcast(float sum, float scaled, float column_scales) {
  asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(sum) : "v"(column_scales), "v"(scaled), "n"(N));
  return sum;
}
template <int kBlock>
__device__ __forceinline__ void fold_block_with_row_broadcast(f32x4& acc, const f32x4& product, float row_scale, float column_scales) {
  acc[0] = fold_one_with_row_broadcast<4 * kBlock + 0>(acc[0], product[0] * row_scale, column_scales);
  acc[1] = fold_one_with_row_broadcast<4 * kBlock + 1>(acc[1], product[1] * row_scale, column_scales);
  acc[2] = fold_one_with_row_broadcast<4 * kBlock + 2>(acc[2], product[2] * row_scale, column_scales);
  acc[3] = fold_one_with_row_broadcast<4 * kBlock + 3>(acc[3], product[3] * row_scale, column_scales);
}
__device__ __forceinline__ void fold_with_row_broadcast(f32x4& acc, const f32x4& product, float row_scale, float column_scales,
                                                        int block) {
  if (block == 0) fold_block_with_row_broadcast<0>(acc, product, row_scale, column_scales);
  else if (block == 1) fold_block_with_row_broadcast<1>(acc, product, row_scale, column_scales);
  else if (block == 2) fold_block_with_row_broadcast<2>(acc, product, row_scale, column_scales);
  else fold_block_with_row_broadcast<3>(acc, product, row_scale, column_scales);
}

// A tile of WM x WN waves, each TM x TN blocks of 16 x 16; a k-tile is one scale
// block (128 bytes of every row) with its row and column scales.  A chunk is
// what one request of every wave fills.  The first kEarly chunks of a k-tile
// have kDepth + 1 slots in LDS, the others and the scales kDepth.
template <int WM_, int WN_, int TM_, int TN_, int kDepth_, int kEarly_>
struct Fp8Tile {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, kDepth = kDepth_, kEarly = kEarly_;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves, kWaveM = 16 * TM, kWaveN = 16 * TN;
  static constexpr int BM = WM * kWaveM, BN = WN * kWaveN, BK = 128, kRowBytes = 128;
  static constexpr int kChunkRows = 8 * kWaves, kChunkBytes = kChunkRows * kRowBytes;
  static constexpr int kChunksA = BM / kChunkRows, kChunks = kChunksA + BN / kChunkRows, kLate = kChunks - kEarly;
  static constexpr int kEarlyBytes = kEarly * kChunkBytes, kLateBytes = kLate * kChunkBytes;
  static constexpr int kLateOffset = (kDepth + 1) * kEarlyBytes, kScaleOffset = kLateOffset + kDepth * kLateBytes;
  // Scales of a k-tile: BM row scales, then BN column scales (or the block scale of every 64 columns, 64 times).
  static constexpr int kScaleRequests = (BM + BN) / 64, kScaleBytes = 256 * kScaleRequests;
  static constexpr int kLdsBytes = kScaleOffset + kDepth * kScaleBytes;
  static constexpr int kPitch = kWaveN * 2 + 16, kRegion = kWaveM * kPitch;  // epilogue staging of a wave, bytes
  static_assert(kLdsBytes <= 160 * 1024 && kWaves * kRegion <= kLdsBytes, "LDS of a compute unit");
  static_assert(BM % kChunkRows == 0 && BN % kChunkRows == 0 && kWaveN % kChunkRows == 0, "whole chunks");
  static_assert(kChunkRows % kWaveM == 0 || kWaveM % kChunkRows == 0, "a wave's rows in whole chunks or in one");
  static_assert(kEarly == kChunks || kEarly <= kChunksA, "operand B is early or late as a whole");
  static_assert(BM % 64 == 0 && BN % 64 == 0 && kScaleRequests <= kWaves && (TN == 2 || TN % 4 == 0), "scales by 64");
  static_assert(kDepth >= 2 && kDepth <= 4, "the waits of the k loop's end");
};

// One output tile at (m0, n0).
//
// The small tiles are bound by the latency of a k-tile where a compute unit has
// one workgroup (a chain of requests, a barrier, fragment reads), by the request
// path (one 1 KB request per 16 cycles: the 32 of a 128 x 128 k-tile last as long
// as its MFMAs) where it has several.  Before, they ran 32 x 32 x 64 MFMAs whose 16
// registers were folded behind the next one's, and their requests left in one go
// behind the last block, held up by one another.  us before / now; the same bits
// unless a run's products span more than 24 bits, where up to 4e-5 of the outputs lie on
// the other side of a bf16 rounding (2-norm from 64-bit sums the same to 1e-6 of it):
//   64 x 64:    48 x 14336, k 4096 12.1 / 10.8   144 x 3840, k 10240 23.4 / 22.0   512 x 4096, k 4096 16.1 / 14.6
//               3000 x 1024 over 1500 tokens, column scales 12.0 / 10.0   1000 x 2048, k 5120 20.1 / 19.1
//   128 x 128:  1000 x 5120, k 2048 18.9 / 16.6   1024 x 4096, k 8192 45.6 / 38.8
//               1024 x 4096 over 8192 tokens, column scales 50.9 / 44.7
template <typename Cfg, bool kColumnScales>
__device__ __forceinline__ void fp8_gemm_tile(const Fp8GemmParams& p, uint8_t* lds_bytes, int64_t m0, int64_t n0) {
  constexpr int TM = Cfg::TM, TN = Cfg::TN, kChunks = Cfg::kChunks, kChunksA = Cfg::kChunksA, kEarly = Cfg::kEarly, kDepth = Cfg::kDepth;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
#ifdef FSH_TRACE
  const uint64_t t_entry = __builtin_amdgcn_s_memrealtime();
#endif
  const int ktiles = static_cast<int>(p.k / Cfg::BK);

  // Load side: request c of a wave fills rows [kChunkRows c + 8 wave, +8) of
  // the tile's operand A, from c = kChunksA on of operand B; lane l fills slot l & 7 of
  // row l >> 3 there.  Rows past the matrix are read from its last row (their
  // products are never stored).
  const int fill_row = lane >> 3;
  const int fill_chunk = (lane & 7) ^ (((8 * wave + fill_row) >> 1) & 7);
  uint32_t voff[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int64_t first = c < kChunksA ? m0 : n0, size = c < kChunksA ? p.m : p.n, ld = c < kChunksA ? p.ldxq : p.ldwq;
    int64_t row = first + Cfg::kChunkRows * (c < kChunksA ? c : c - kChunksA) + 8 * wave + fill_row;
    row = row < size ? row : size - 1;
    voff[c] = static_cast<uint32_t>((row - first) * ld + fill_chunk * 16);
  }
  const uint8_t* Ab = uniform_ptr(p.xq + m0 * p.ldxq);
  const uint8_t* Bb = uniform_ptr(p.wq + n0 * p.ldwq);
  typedef __attribute__((address_space(3))) uint8_t* lds_address;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_address)lds_bytes));
  const uint32_t fill_lds = lds_base + static_cast<uint32_t>(wave * 1024);
  // Where a k-tile lies: the offsets of its early chunks, of its late ones and of its scales.
  struct Place {
    int early, late, scales;
  };
  constexpr Place kFirst{0, Cfg::kLateOffset, Cfg::kScaleOffset};
  constexpr Place kLast{kDepth * Cfg::kEarlyBytes, Cfg::kLateOffset + (kDepth - 1) * Cfg::kLateBytes,
                        Cfg::kScaleOffset + (kDepth - 1) * Cfg::kScaleBytes};
  const auto place_after = [](const Place& at) {
    return Place{at.early == kLast.early ? kFirst.early : at.early + Cfg::kEarlyBytes,
                 at.late == kLast.late ? kFirst.late : at.late + Cfg::kLateBytes,
                 at.scales == kLast.scales ? kFirst.scales : at.scales + Cfg::kScaleBytes};
  };
  auto request = [&](int kt, const Place& at, int c) {
    dma_load_16(voff[c], (c < kChunksA ? Ab : Bb) + static_cast<int64_t>(kt) * Cfg::kRowBytes,
                fill_lds + (c < kEarly ? at.early : at.late), (c < kEarly ? c : c - kEarly) * Cfg::kChunkBytes);
  };
  // The first k-tile's operands, ahead of everything that has to be worked out
  // for the scales (behind it, a tile of one k-tile took 0.02 to 0.05 us longer:
  // us of 6194 x 10880 over 100 tokens, before the chunks / behind / ahead 34.9 /
  // 35.4 / 35.0; 300 x 2048, k 2048 7.9 / 6.9 / 6.8).
  Place ahead = kFirst;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) request(0, ahead, c);
  // The scales of a k-tile ride the same global->LDS path, 64 by one request of
  // each wave: the row scales, then the column scales -- or the block scale of
  // 64 of the tile's columns, 64 times.  (A load that the compiler sees inside
  // the loop makes it wait for all requests in flight.)  Waves past the
  // requests repeat the first ones.
  const int scale_request = wave % Cfg::kScaleRequests;
  const float* scale_src = p.xs;
  int64_t scale_step = p.m;
  uint32_t scale_voff = 0;
  if (scale_request < Cfg::BM / 64) {
    const int64_t row = m0 + scale_request * 64 + lane;
    scale_voff = static_cast<uint32_t>((row < p.m ? row : p.m - 1) * 4);
  } else {
    const int64_t first = n0 + (scale_request - Cfg::BM / 64) * 64;
    if (kColumnScales) {
      scale_voff = static_cast<uint32_t>((first + lane < p.n ? first + lane : p.n - 1) * 4);
      scale_src = p.cs;
      scale_step = p.n;
    } else {
      const int64_t block = first / 128, last = (p.n - 1) / 128;
      scale_src = p.ws + (block < last ? block : last) * p.ws_cb;
      scale_step = p.ws_kb;
    }
  }
  const uint32_t scale_lds = lds_base + scale_request * 256;
  auto request_scales = [&](int kt, const Place& at) {
    dma_touch_4(scale_voff, reinterpret_cast<const uint8_t*>(scale_src + kt * scale_step), scale_lds + at.scales);
  };

  request_scales(0, ahead);
  ahead = place_after(ahead);

  // Fragment side: row = lane & 15 of a 16-row block, chunks g and g + 4 of its
  // eight (g = lane / 16), each in slot chunk ^ ((row >> 1) & 7).  Any split of
  // the 128 bytes over the four g will do that both operands share; with chunks
  // 2 g and 2 g + 1 the reads met in the banks (25 % of the kernel's cycles by
  // the counter: the LDS serves a 16-byte read to lanes of two neighbouring g at
  // a time, whose slots stay apart if their chunks differ in bit 0).
  const int frag_row = lane & 15, group = lane >> 4;
  uint32_t frag_off[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    frag_off[c] = static_cast<uint32_t>(frag_row * Cfg::kRowBytes + (((group + 4 * c) ^ ((frag_row >> 1) & 7)) * 16));
  // `row` of the rows that start at `chunk`
  auto read_frag = [&](int chunk, int row) -> v8i32 {
    const uint8_t* base = lds_bytes + chunk + row * Cfg::kRowBytes;
    const u32x4 lo = *reinterpret_cast<const u32x4*>(base + frag_off[0]);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(base + frag_off[1]);
    return v8i32{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z), static_cast<int>(lo.w),
                 static_cast<int>(hi.x), static_cast<int>(hi.y), static_cast<int>(hi.z), static_cast<int>(hi.w)};
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The rest of the first kDepth - 1 k-tiles and the early chunks of the next.
  Place now = kFirst, before = kLast;  // of k-tile kt and of the one before it, whose slots are free
#pragma unroll
  for (int kt = 1; kt < kDepth; ++kt) {
    if (kt < ktiles) {
      if (kt + 1 < kDepth) request_scales(kt, ahead);
#pragma unroll
      for (int c = 0; c < kChunks; ++c)
        if (kt + 1 < kDepth || c < kEarly) request(kt, ahead, c);
    }
    ahead = place_after(ahead);
  }
  constexpr int kRequests = kChunks + 1;  // of a k-tile, per wave
  if (ktiles >= kDepth) wait_for_dma_loads_but<kEarly + (kDepth - 2) * kRequests>();
  else if (kDepth >= 4 && ktiles == 3) wait_for_dma_loads_but<2 * kRequests>();
  else if (kDepth >= 3 && ktiles == 2) wait_for_dma_loads_but<kRequests>();
  else wait_for_dma_loads();
  asm volatile("s_barrier" ::: "memory");

#ifdef FSH_TRACE
  // Time per phase of the k loop, summed over the k-tiles (10 ns ticks).
  uint64_t t_compute = 0, t_wait = 0, t_barrier = 0, t_mark = __builtin_amdgcn_s_memrealtime();
  const uint64_t t_begin = t_mark;
  auto lap = [&](uint64_t& sum) {
    const uint64_t now = __builtin_amdgcn_s_memrealtime();
    sum += now - t_mark;
    t_mark = now;
  };
#endif
  // The k loop is rotated by a column of blocks: the barrier that hands over
  // k-tile kt + 1 sits before the last column of k-tile kt, and behind each of
  // its MFMAs the wave reads the fragment of kt + 1 that takes the place of the
  // one just used.
  //   carried into a k-tile: afrag, bfrag[0]
  // Behind that barrier the slots of k-tile kt are free: in k-tile kt + 1 they
  // take the scales and late chunks of kt + kDepth, then the early ones of
  // kt + kDepth + 1, one request behind every few MFMAs.
  constexpr int kBlocks = TM * TN;
  v8i32 afrag[TM], bfrag[2];
  constexpr int kScaleRegs = (TN + 3) / 4, kBlocksPerReg = TN < 4 ? TN : 4;
  float s[TM], cs_rows[kScaleRegs];
  // Row scales of the wave's rows for k-tile kt, times the block scale in the
  // block-scale variant; a lane owns output row lane & 15 of each of its blocks.
  auto read_scales = [&](const Place& at) {
    const float* rows = reinterpret_cast<const float*>(lds_bytes + at.scales);
#pragma unroll
    for (int i = 0; i < TM; ++i) s[i] = rows[wm * Cfg::kWaveM + i * 16 + frag_row];
    if (kColumnScales) {
      // Register q holds, in every row of 16 lanes, the 16 scales that the lanes
      // of that row fold column blocks 4 q .. 4 q + 3 with: lane 4 b + r of the
      // row the scale of accumulator r of block 4 q + b.  A fold takes it through
      // the data-parallel-primitive broadcast of the multiply-add itself.
#pragma unroll
      for (int q = 0; q < kScaleRegs; ++q)
        cs_rows[q] = rows[Cfg::BM + wn * Cfg::kWaveN + q * 64 + 16 * (((lane & 15) >> 2) % kBlocksPerReg) + 4 * group + (lane & 3)];
    } else {
      const float block_scale = rows[Cfg::BM + wn * Cfg::kWaveN];
#pragma unroll
      for (int i = 0; i < TM; ++i) s[i] *= block_scale;
    }
  };
  // The wave's rows of A lie in whole chunks, or in a part of one; those of B in whole chunks.
  const int a_chunk = wm * Cfg::kWaveM / Cfg::kChunkRows, a_row = wm * Cfg::kWaveM % Cfg::kChunkRows;
  const int b_chunk = kChunksA + wn * Cfg::kWaveN / Cfg::kChunkRows;
  const auto chunk_at = [](const Place& at, int c, bool early) {
    return (early ? at.early : at.late) + (early ? c : c - kEarly) * Cfg::kChunkBytes;
  };
  auto read_a = [&](const Place& at, int i) {
    const int c = a_chunk + i * 16 / Cfg::kChunkRows;
    afrag[i] = read_frag(chunk_at(at, c, c < kEarly), a_row + i * 16 % Cfg::kChunkRows);
  };
  auto read_b = [&](const Place& at, int j) {
    bfrag[j & 1] = read_frag(chunk_at(at, b_chunk + j * 16 / Cfg::kChunkRows, kEarly == kChunks), j * 16 % Cfg::kChunkRows);
  };
  constexpr bool kWholeAhead = TN == 2;
  read_b(now, 0);
  if (kWholeAhead) read_b(now, 1);
#pragma unroll
  for (int i = 0; i < TM; ++i) read_a(now, i);

  // The MFMA that request r of a k-tile goes out behind, the late chunks first
  // and closer together: with kDepth = 2 the last of them has the rest of this
  // k-tile to arrive.  All go out before the wait for the next k-tile.
  constexpr auto behind_mfma = [](int r) {
    if (kBlocks < 2 * kChunks) return r * (kBlocks - TM) / kChunks;
    const int span = kBlocks / kChunks, late_span = span - 1 > 0 ? span - 1 : 1;
    return r < Cfg::kLate ? r * late_span : Cfg::kLate * late_span + (r - Cfg::kLate) * span;
  };
  static_assert(behind_mfma(kChunks - 1) < kBlocks - TM, "the count that the wait leaves in flight");
  // more: k-tile kt + 1 exists; late, early: kt + kDepth - 1 and kt + kDepth do, and their late and early
  // chunks go out.  Tags, so that no request sits behind a branch of its own.
  auto k_tile = [&](int kt, auto more_tag, auto late_tag, auto early_tag) {
    constexpr bool more = decltype(more_tag)::value, late = decltype(late_tag)::value, early = decltype(early_tag)::value;
    const Place next = place_after(now);
    // The scales are first needed by the first fold, kLag blocks in.
    read_scales(now);
    // The wave's 16x16 blocks, column by column.  One 16x16x128 MFMA gives a
    // block's partial product for this scale block; it is folded into the result
    // (4 fused multiply-adds, or multiply + fused multiply-add with per-column
    // scales) kLag blocks later: a fold that reads the product of an MFMA issued
    // just before it waits for the matrix core to drain.
    constexpr int kLag = kBlocks > 8 ? 4 : 2;
    f32x4 part[kLag + 1];
    auto fold = [&](int blk) {
      const int pi = blk % TM, pj = blk / TM;
      const f32x4& product = part[blk % (kLag + 1)];
      if (kColumnScales) {
        fold_with_row_broadcast(acc[pi][pj], product, s[pi], cs_rows[pj / 4], pj % 4);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[pi][pj][r] = __builtin_fmaf(product[r], s[pi], acc[pi][pj][r]);
      }
      // An empty statement that "uses" the folded block keeps its arithmetic
      // on this side of the next scheduling barrier.
      asm volatile("" : "+v"(acc[pi][pj]));
    };
#pragma unroll
    for (int blk = 0; blk < kBlocks; ++blk) {
      const int i = blk % TM, j = blk / TM;
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      if (blk == kBlocks - TM) {
        // Every fragment of this k-tile is in registers: hand its slots over.
#ifdef FSH_TRACE
        lap(t_compute);
#endif
        // This wave's part of k-tile kt + 1 has landed; what was requested behind it stays in flight.
        if (early) wait_for_dma_loads_but<kEarly + (kDepth - 2) * kRequests>();
        else if (kDepth >= 4 && kt + 4 == ktiles) wait_for_dma_loads_but<2 * kRequests>();
        else if (kDepth >= 3 && kt + 3 == ktiles) wait_for_dma_loads_but<kRequests>();
        else if (more) wait_for_dma_loads();
#ifdef FSH_TRACE
        lap(t_wait);
#endif
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#ifdef FSH_TRACE
        lap(t_barrier);
#endif
      }
      // The next column's B fragment, a column ahead (of two columns both come with the k-tile's first ones).
      if (!kWholeAhead && i == 0 && j + 1 < TN) read_b(now, j + 1);
      // Wave priority falls as the k-tile proceeds: of the two waves of a SIMD
      // the one that is behind wins the issue slot, so both reach the barrier
      // together (with equal priorities the older wave runs ahead and then
      // idles at the barrier while the other finishes alone, without a
      // partner to overlap its folds with).
      if (blk * 4 == 0 * kBlocks) __builtin_amdgcn_s_setprio(3);
      if (blk * 4 == 1 * kBlocks) __builtin_amdgcn_s_setprio(2);
      if (blk * 4 == 2 * kBlocks) __builtin_amdgcn_s_setprio(1);
      if (blk * 4 == 3 * kBlocks) __builtin_amdgcn_s_setprio(0);
      part[blk % (kLag + 1)] =
          __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bfrag[j & 1], afrag[i], zero, 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (blk >= kBlocks - TM && more) {  // what the next k-tile starts with
        if (i == 0) read_b(next, 0);
        read_a(next, i);
        if (kWholeAhead && blk == kBlocks - 1) read_b(next, 1);
      }
      if (late && blk == 0) request_scales(kt + kDepth - 1, before);
#pragma unroll
      for (int r = 0; r < kChunks; ++r)
        if (blk == behind_mfma(r)) {
          if (r < Cfg::kLate) {
            if (late) request(kt + kDepth - 1, before, kEarly + r);
          } else if (early) {
            request(kt + kDepth, before, r - Cfg::kLate);
          }
        }
      if (blk >= kLag) fold(blk - kLag);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int blk = kBlocks - kLag; blk < kBlocks; ++blk) fold(blk);
    before = now;
    now = next;
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  int kt = 0;
  for (; kt + kDepth < ktiles; ++kt) k_tile(kt, yes, yes, yes);
  if (kDepth <= ktiles) k_tile(kt++, yes, yes, no);
  for (; kt + 1 < ktiles; ++kt) k_tile(kt, yes, no, no);
  k_tile(ktiles - 1, no, no, no);
#ifdef FSH_TRACE
  if (p.schedule.trace && lane == 0) {
    uint64_t* out = p.schedule.trace + (static_cast<int64_t>(blockIdx.x) * Cfg::kWaves + wave) * 8;
    out[0] = t_begin; out[1] = t_compute; out[2] = t_wait; out[3] = t_barrier; out[4] = t_mark; out[5] = t_entry;
  }
#endif

  // Epilogue: bf16 finals to the wave's staging region as [row][col], then
  // 16-byte row stores, rows and 8-column groups past the matrix skipped.
  uint8_t* region = lds_bytes + wave * Cfg::kRegion;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<u32x2*>(region + (i * 16 + frag_row) * Cfg::kPitch + (j * 16 + 4 * group) * 2) =
          u32x2{pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
  wave_lds_sync();
  store_fp8_product<Cfg::kWaveM, Cfg::kWaveN, Cfg::kPitch>(region, p, m0 + wm * Cfg::kWaveM, n0 + wn * Cfg::kWaveN, lane);
#ifdef FSH_TRACE
  if (p.schedule.trace && lane == 0) {
    __builtin_amdgcn_s_waitcnt(0);
    p.schedule.trace[(static_cast<int64_t>(blockIdx.x) * Cfg::kWaves + wave) * 8 + 6] = __builtin_amdgcn_s_memrealtime();
    uint32_t hw_id;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw_id));
    uint32_t xcc_id;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc_id));
    p.schedule.trace[(static_cast<int64_t>(blockIdx.x) * Cfg::kWaves + wave) * 8 + 7] = (static_cast<uint64_t>(xcc_id) << 32) | hw_id;
  }
#endif
}

template <typename Cfg, bool kColumnScales, int kBlocksPerUnit>
__global__ __launch_bounds__(Cfg::kThreads, kBlocksPerUnit * Cfg::kWaves / 4) void fp8_gemm_tiles_kernel(const Fp8GemmParams p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  int64_t unused_batch;
  int tm, tn;
  if (!tile_of_workgroup(p.schedule, blockIdx.x, &unused_batch, &tm, &tn)) return;  // whole workgroup
  fp8_gemm_tile<Cfg, kColumnScales>(p, lds_bytes, static_cast<int64_t>(uniform_i32(tm)) * Cfg::BM,
                                    static_cast<int64_t>(uniform_i32(tn)) * Cfg::BN);
}

}  // namespace
}  // namespace fsh
