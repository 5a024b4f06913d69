// Forward GEMM of a linear layer whose weight arrives already quantized
// (128x128 tiles, FP8 E4M3FN) from the bucket unpack: 1x128 quantization of
// the activation and the FP8 product with both sets of scales.
//
//   xq, xs = quantize each run of 128 consecutive elements of a row of x
//            (amax floored at 1e-12, scale = fp32(448 / fp64(amax)),
//            q = e4m3fn(fp32(x) * scale), stored scale = 1.0f / scale)
//   out[m][n] = bf16( sum over k-blocks kb of
//                     dot(xq[m][kb], wq[n][kb]) * (xs[kb][m] * ws[n / 128][kb]) )
//
// Matrix cores: v_mfma_f32_16x16x128_f8f6f4 here, 32x32x64 in the smaller tiles
// (twice the rate of the 32x32x16 FP8 form on gfx950).  A k-tile is one scale
// block (128 bytes of each row), so its partial products are accumulated from
// zero in a scratch accumulator and folded into the result with one fused
// multiply-add per element; the folds of one block run on the vector ALU while
// the matrix core works on the next ones.
#include "fp8_tiles.hpp"

namespace fsh {
namespace {

// ------------------------------------------------------------ 1x128 quantize
// A workgroup owns 16 rows x 512 columns (4 scale blocks per row).  Sixteen
// lanes own one run of 128 elements (16 bytes each); a wavefront load covers
// four runs = 1 KB of one row.  All four loads of a thread are issued before
// the first is used.  The maximum of a run stays inside its row of 16 lanes
// (four DPP steps, no LDS, no barrier).  Scales go through LDS so that they
// leave as 64-byte runs of the [k-block][row] table.
//
// Bound by memory when large, by the chain of one thread's passes (each with
// two divisions) when small.  With 64 rows per workgroup, sixteen passes (us,
// 64 / 16 / 4 rows):  48 x 4096 5.5 / 4.2 / 4.0   1000 x 2048 7.5 / 4.1 / 4.0
//   2048 x 4096 9.1 / 6.1 / 6.8   8192 x 4096 22.7 / 18.6 / 19.0   8192 x 14336 61.1 / 57.3 / 61.4
constexpr int kActThreads = 256;
constexpr int kActRows = 16;
constexpr int kActBlocks = 4;  // 128-element runs per row and workgroup
constexpr int kActPasses = kActRows * kActBlocks * 16 / kActThreads;

struct ActQuantParams {
  const uint8_t* x;
  uint8_t* q;
  float* scales;
  int64_t rows, cols, ldx, ldq;  // elements; ldq = cols rounded up to 128
  int64_t first_row;             // of this launch
  int32_t col_groups;            // ceil(ceil(cols / 128) / 4)
  float eps;
};

__global__ __launch_bounds__(kActThreads) void act_quant_1x128_kernel(const ActQuantParams p) {
  __shared__ float lds_scales[kActBlocks * kActRows];
  const int tid = threadIdx.x;
  const int sub = tid & 15, run_lane = tid >> 4;
  const int64_t tile_r = blockIdx.x / p.col_groups, tile_c = blockIdx.x % p.col_groups;
  const int64_t row0 = p.first_row + tile_r * kActRows, kb0 = tile_c * kActBlocks;

  u32x4 v[kActPasses];
#pragma unroll
  for (int pass = 0; pass < kActPasses; ++pass) {
    const int run = pass * 16 + run_lane;  // within the tile
    const int64_t row = row0 + run / kActBlocks;
    const int64_t col = (kb0 + run % kActBlocks) * 128 + sub * 8;
    v[pass] = u32x4{0, 0, 0, 0};
    if (row < p.rows && col < p.cols) v[pass] = load_stream_u32x4(p.x + (row * p.ldx + col) * 2);
  }
#pragma unroll
  for (int pass = 0; pass < kActPasses; ++pass) {
    const int run = pass * 16 + run_lane;
    const int64_t row = row0 + run / kActBlocks;
    const int64_t col = (kb0 + run % kActBlocks) * 128 + sub * 8;
    uint32_t m = pk_max_u16(v[pass].x & 0x7FFF7FFFu, v[pass].y & 0x7FFF7FFFu);
    m = pk_max_u16(m, v[pass].z & 0x7FFF7FFFu);
    m = pk_max_u16(m, v[pass].w & 0x7FFF7FFFu);
    const uint32_t lo = m & 0xFFFFu, hi = m >> 16;
    m = row16_max_u32(lo > hi ? lo : hi);
    float scale, recip;
    tile_scale(bf16_bits_to_f32(m), p.eps, scale, recip);
    if (sub == 0) lds_scales[(run % kActBlocks) * kActRows + run / kActBlocks] = recip;
    if (row < p.rows && col < p.ldq) {
      const uint32_t d[4] = {v[pass].x, v[pass].y, v[pass].z, v[pass].w};
      uint32_t w[2] = {0, 0};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e0 = u32_as_f32(d[j] << 16) * scale;
        const float e1 = u32_as_f32(d[j] & 0xFFFF0000u) * scale;
        w[j >> 1] = cvt2_fp8(e0, e1, w[j >> 1], (j & 1) != 0);
      }
      store_stream_u32x2(p.q + row * p.ldq + col, w[0], w[1]);
    }
  }
  __syncthreads();
  if (tid < kActBlocks * kActRows) {
    const int kbl = tid / kActRows, r = tid % kActRows;
    const int64_t kb = kb0 + kbl, row = row0 + r;
    if (row < p.rows && kb * 128 < p.ldq) p.scales[kb * p.rows + row] = lds_scales[tid];
  }
}

// ----------------------------------------------------------------- FP8 GEMM
// 256 x 256 output tile per workgroup (262 flop per operand byte, which is
// what keeps the request rate to L2 within reach at FP8 speed), eight waves of
// 64 x 128 (four by eight 16x16 blocks).  A wave's 128 accumulators stay in
// architectural VGPRs, where the vector ALU folds into them, and two waves
// share a SIMD, so one wave's folds run under the other's MFMAs.  Operand
// tiles are 128 bytes per row and k-tile and travel global -> LDS directly,
// 16-byte chunk c of row r in slot c ^ ((r >> 1) & 7).
//
// Bound by power, and with column scales by the vector ALU as well (two
// operations per element and k-block).  What the parts cost, us of 8192 x 14336,
// k 4096 (404), and of its weight gradient (449): without the requests of the
// loop 315 and 390, with operands that stay in L2 367 and 422, without the
// fragment reads 378 and 397, without the folds 367 and 340.
//
// A 16x16x128 MFMA is a block's whole product of a k-tile: four registers
// that a fold can follow four blocks later.  LDS holds two k-tiles and three
// eighths of a third, in chunks of 64 rows, so that the requests of a k-tile
// leave one by one behind its MFMAs.  In two 64 KB stages they had to leave in
// half of it: they then ask for all that the request path can take (64 of 16
// cycles in 1024), and the last were waited for.  One round of k-tiles on the same
// card, us before / with the chunks (same bits): forward 4096 x 4096 110 / 110,
// 14336 x 4096 419 / 403, 4096 x 14336 399 / 370, 1024 x 4096 (half tiles) 39.3 / 34.2;
// weight gradients 122 / 121, 455 / 441, 449 / 437.  The scales of a k-tile take one 4-byte
// request of each wave; the block scales had a window of 256 k-tiles of their own
// and an instantiation that refilled it.
//
// TM_ = 1 is the half tile (128 x 256, waves of 32 x 128) that the tiles of a
// last, at most half-full round are cut into.
template <int TM_>
struct Fp8GemmCfg {
  static constexpr int BM = 128 * TM_, BN = 256, BK = 128, WM = 4, WN = 2;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves, kWaveM = BM / WM, kWaveN = BN / WN;
  static constexpr int TM = kWaveM / 16, TN = kWaveN / 16;  // blocks of 16 x 16 per wave
  static constexpr int kRowBytes = 128;
  // A chunk is what one request of every wave fills: 64 rows of an operand.
  static constexpr int kChunkRows = 8 * kWaves, kChunkBytes = kChunkRows * kRowBytes;       // 8 KB
  static constexpr int kChunksA = BM / kChunkRows, kChunks = kChunksA + BN / kChunkRows;    // per k-tile: 8 (6)
  // LDS holds 19: the early chunks of a k-tile, the first of operand A (all of
  // a half tile's), have three slots each and are requested a k-tile ahead of
  // the late ones, which have two.
  static constexpr int kSlots = 19;
  static constexpr int kEarly = kSlots - 2 * kChunks < kChunks ? kSlots - 2 * kChunks : kChunks, kLate = kChunks - kEarly;
  static constexpr int kEarlyBytes = kEarly * kChunkBytes, kLateBytes = kLate * kChunkBytes;
  static constexpr int kLateOffset = 3 * kEarlyBytes;
  static constexpr int kPitch = kWaveN * 2 + 16;               // epilogue staging, bytes
  static constexpr int kRegion = kWaveM * kPitch;              // per wave
  // Two stages of scales: 256 row scales, then 256 column scales (or the two
  // block scales, 64 times each).
  static constexpr int kScaleOffset = kSlots * kChunkBytes, kScaleStageBytes = 2048;
  static constexpr int kLdsBytes = kScaleOffset + 2 * kScaleStageBytes;
  static_assert(kLdsBytes <= 160 * 1024 && kWaves * kRegion <= kLdsBytes, "LDS of a compute unit");
  static_assert(kEarly > 0 && 3 * kEarly + 2 * kLate <= kSlots, "two k-tiles and a part of the next");
};
using Fp8Gemm = Fp8GemmCfg<2>;

// One output tile (TM_ = 2) or half tile (TM_ = 1, rows [128 half, +128) of the tile).
template <bool kColumnScales, int TM_>
__device__ __forceinline__ void fp8_gemm_tile(const Fp8GemmParams& p, uint8_t* lds_bytes, int tm, int tn, int half) {
  using Cfg = Fp8GemmCfg<TM_>;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, kChunks = Cfg::kChunks, kChunksA = Cfg::kChunksA, kEarly = Cfg::kEarly;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int64_t m0 = static_cast<int64_t>(tm) * Fp8Gemm::BM + static_cast<int64_t>(half) * Cfg::BM;
  const int64_t n0 = static_cast<int64_t>(tn) * Cfg::BN;
  if (m0 >= p.m) return;  // the second half of a tile that ends in its first (whole workgroup)
#ifdef FSH_TRACE
  const uint64_t t_entry = __builtin_amdgcn_s_memrealtime();
#endif
  const int ktiles = static_cast<int>(p.k / Cfg::BK);

  // Load side: request c of a wave fills rows [64 c + 8 wave, +8) of the tile's
  // operand A, from c = kChunksA on of operand B; lane l fills slot l & 7 of
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
  // Where a k-tile lies: the offsets of its early chunks and of its late ones.
  struct Place {
    int early, late;
  };
  const auto place_after = [](const Place& at) {
    return Place{at.early == 2 * Cfg::kEarlyBytes ? 0 : at.early + Cfg::kEarlyBytes,
                 at.late == Cfg::kLateOffset ? Cfg::kLateOffset + Cfg::kLateBytes : Cfg::kLateOffset};
  };
  auto request = [&](int kt, const Place& at, int c) {
    dma_load_16(voff[c], (c < kChunksA ? Ab : Bb) + static_cast<int64_t>(kt) * Cfg::kRowBytes,
                fill_lds + (c < kEarly ? at.early : at.late), (c < kEarly ? c : c - kEarly) * Cfg::kChunkBytes);
  };
  // The scales of a k-tile ride the same global->LDS path: 64 row scales by
  // each of the first four waves, 64 column scales by each of the others -- or
  // by two of them each the block scale of 128 of the tile's columns, 64 times.
  // (A load that the compiler sees inside the loop makes it wait for all
  // requests in flight.)
  const float* scale_src = p.xs;
  int64_t scale_step = p.m;
  uint32_t scale_voff = 0, scale_slot = wave % (Cfg::BM / 64);
  if (wave < 4) {
    const int64_t row = m0 + scale_slot * 64 + lane;
    scale_voff = static_cast<uint32_t>((row < p.m ? row : p.m - 1) * 4);
  } else if (kColumnScales) {
    const int64_t col = n0 + (wave - 4) * 64 + lane;
    scale_voff = static_cast<uint32_t>((col < p.n ? col : p.n - 1) * 4);
    scale_src = p.cs;
    scale_step = p.n;
    scale_slot = wave;
  } else {
    const int64_t block = n0 / 128 + (wave >> 1 & 1), last = (p.n - 1) / 128;
    scale_src = p.ws + (block < last ? block : last) * p.ws_cb;
    scale_step = p.ws_kb;
    scale_slot = 4 + (wave >> 1 & 1);
  }
  const uint32_t scale_lds = lds_base + Cfg::kScaleOffset + scale_slot * 256;
  auto request_scales = [&](int kt) {
    dma_touch_4(scale_voff, reinterpret_cast<const uint8_t*>(scale_src + kt * scale_step), scale_lds + (kt & 1) * Cfg::kScaleStageBytes);
  };

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

  // The first k-tile and the early chunks of the second.
  Place now{0, Cfg::kLateOffset};  // of k-tile kt
  request_scales(0);
#pragma unroll
  for (int c = 0; c < kChunks; ++c) request(0, now, c);
  if (ktiles > 1) {
#pragma unroll
    for (int c = 0; c < kEarly; ++c) request(1, place_after(now), c);
    wait_for_dma_loads_but<kEarly>();
  } else {
    wait_for_dma_loads();
  }
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
  // Behind that barrier the slots of k-tile kt are free: in k-tile kt + 1 the
  // late chunks of kt + 2 go out, then the early ones of kt + 3, one request
  // behind every few MFMAs.
  constexpr int kBlocks = TM * TN;
  v8i32 afrag[TM], bfrag[2];
  constexpr int kScaleRegs = TN / 4;
  float s[TM], cs_rows[kScaleRegs];
  // Row scales of the wave's rows for k-tile kt, times the block scale in the
  // block-scale variant; a lane owns output row lane & 15 of each of its blocks.
  auto read_scales = [&](int kt) {
    const float* rows = reinterpret_cast<const float*>(lds_bytes + Cfg::kScaleOffset + (kt & 1) * Cfg::kScaleStageBytes);
#pragma unroll
    for (int i = 0; i < TM; ++i) s[i] = rows[wm * Cfg::kWaveM + i * 16 + frag_row];
    if (kColumnScales) {
      // Register q holds, in every row of 16 lanes, the 16 scales that the lanes
      // of that row fold column blocks 4 q .. 4 q + 3 with: lane 4 b + r of the
      // row the scale of accumulator r of block 4 q + b.  A fold takes it through
      // the data-parallel-primitive broadcast of the multiply-add itself.
#pragma unroll
      for (int q = 0; q < kScaleRegs; ++q)
        cs_rows[q] = rows[256 + wn * Cfg::kWaveN + q * 64 + 16 * ((lane & 15) >> 2) + 4 * group + (lane & 3)];
    } else {
      const float block_scale = rows[256 + wn * 64];
#pragma unroll
      for (int i = 0; i < TM; ++i) s[i] *= block_scale;
    }
  };
  // The chunk of the wave's rows of A (waves of 32 rows share one) and its two of B.
  const int a_chunk = wm * Cfg::kWaveM / Cfg::kChunkRows, a_row = wm * Cfg::kWaveM % Cfg::kChunkRows;
  const bool a_early = a_chunk < kEarly;
  const int a_from = (a_early ? a_chunk : a_chunk - kEarly) * Cfg::kChunkBytes + a_row * Cfg::kRowBytes;
  constexpr bool kBEarly = kEarly == kChunks;
  static_assert(kBEarly || kEarly <= kChunksA, "operand B is early or late as a whole");
  const int b_from = (kChunksA + wn * 2 - (kBEarly ? 0 : kEarly)) * Cfg::kChunkBytes;
  auto read_a = [&](const Place& at, int i) { afrag[i] = read_frag((a_early ? at.early : at.late) + a_from, i * 16); };
  auto read_b = [&](const Place& at, int j) { bfrag[j & 1] = read_frag((kBEarly ? at.early : at.late) + b_from, j * 16); };
  read_b(now, 0);
#pragma unroll
  for (int i = 0; i < TM; ++i) read_a(now, i);

  // more: k-tile kt + 1 exists, and its late chunks go out; more2: kt + 2 exists, and its early ones do.
  // Tags, so that no request sits behind a branch of its own.
  auto k_tile = [&](int kt, auto more_tag, auto more2_tag) {
    constexpr bool more = decltype(more_tag)::value, more2 = decltype(more2_tag)::value;
    const Place next = place_after(now), after = place_after(next);
    // The scales are first needed by the first fold, kLag blocks in.
    read_scales(kt);
    // The wave's 16x16 blocks, column by column.  One 16x16x128 MFMA gives a
    // block's partial product for this scale block; it is folded into the result
    // (4 fused multiply-adds, or multiply + fused multiply-add with per-column
    // scales) kLag blocks later: a fold that reads the product of an MFMA issued
    // just before it waits for the matrix core to drain.
    constexpr int kLag = 4;
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
        // this wave's part of k-tile kt + 1 has landed; the early chunks of kt + 2 stay in flight
        if (more2) wait_for_dma_loads_but<kEarly>();
        else if (more) wait_for_dma_loads();
#ifdef FSH_TRACE
        lap(t_wait);
#endif
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#ifdef FSH_TRACE
        lap(t_barrier);
#endif
      }
      // The next column's B fragment, a column ahead.
      if (i == 0 && j + 1 < TN) read_b(now, j + 1);
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
      }
      // One request behind every few MFMAs, those of the next k-tile first: the
      // last of them has the rest of this k-tile to arrive.
      if (more && blk == 0) request_scales(kt + 1);
#pragma unroll
      for (int r = 0; r < kChunks; ++r) {
        constexpr int kLate = Cfg::kLate;
        if (r < kLate && more && blk == 3 * r) request(kt + 1, next, kEarly + r);
        if (r >= kLate && more2 && blk == 3 * kLate + (r - kLate) * TM) request(kt + 2, after, r - kLate);
      }
      if (blk >= kLag) fold(blk - kLag);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int blk = kBlocks - kLag; blk < kBlocks; ++blk) fold(blk);
    now = next;
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (int kt = 0; kt + 2 < ktiles; ++kt) k_tile(kt, yes, yes);
  if (ktiles > 1) k_tile(ktiles - 2, yes, no);
  k_tile(ktiles - 1, no, no);
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

// kColumnScales = false: the second operand carries one scale per 128 x 128
// tile (a prequantized weight, either orientation).  true: one scale per
// output column and k-block (an operand quantized in 128 x 1 runs).
template <bool kColumnScales>
__global__ __launch_bounds__(Fp8Gemm::kThreads) void fp8_gemm_blockwise_kernel(const Fp8GemmParams p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  int64_t unused_batch;
  int tm, tn;
  if (static_cast<int64_t>(blockIdx.x) < p.whole_grid) {
    if (!tile_of_workgroup(p.schedule, blockIdx.x, &unused_batch, &tm, &tn)) return;  // whole workgroup
    fp8_gemm_tile<kColumnScales, 2>(p, lds_bytes, uniform_i32(tm), uniform_i32(tn), 0);
  } else {
    // Same split over the XCDs as the whole tiles: the two halves of a tile are
    // neighbours in an XCD's run and share the tile's second operand in its L2.
    const int64_t id = static_cast<int64_t>(blockIdx.x) - p.whole_grid;
    const int64_t item = (id % kXcds) * p.half_items_per_xcd + id / kXcds;
    if (item >= p.half_items) return;
    tile_in_order(p.schedule, static_cast<int>(p.schedule.work_items + item / 2), &tm, &tn);
    fp8_gemm_tile<kColumnScales, 1>(p, lds_bytes, uniform_i32(tm), uniform_i32(tn), uniform_i32(static_cast<int>(item & 1)));
  }
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_act_quant_1x128(const void* x_dev, int64_t rows, int64_t cols, int64_t ldx, void* q_dev,
                                int64_t ldq, float* scales_dev, int32_t eps_mode, void* stream) {
  using namespace fsh;
  if (rows < 0 || cols < 0) return fail(FSH_EINVAL, "fsh_act_quant_1x128: negative shape");
  if (rows == 0 || cols == 0) return FSH_OK;
  if (!x_dev || !q_dev || !scales_dev) return fail(FSH_EINVAL, "fsh_act_quant_1x128: null pointer");
  if (eps_mode != FSH_EPS_INPUT_DTYPE && eps_mode != FSH_EPS_FP32)
    return fail(FSH_EINVAL, "fsh_act_quant_1x128: unknown eps_mode %d", eps_mode);
  const int64_t padded = ceil_div(cols, (int64_t)128) * 128;
  if (ldx < cols || ldq != padded)
    return fail(FSH_EINVAL, "fsh_act_quant_1x128: ldx %lld < cols %lld, or ldq %lld is not cols rounded up to 128 (%lld)",
                (long long)ldx, (long long)cols, (long long)ldq, (long long)padded);
  if (cols % 8 || ldx % 8 || !aligned(x_dev, 16) || !aligned(q_dev, 8) || !aligned(scales_dev, 4))
    return fail(FSH_ENOTSUP, "fsh_act_quant_1x128: cols and ldx must be multiples of 8, x 16-byte and q 8-byte aligned");
  ActQuantParams p;
  p.x = static_cast<const uint8_t*>(x_dev);
  p.q = static_cast<uint8_t*>(q_dev);
  p.scales = scales_dev;
  p.rows = rows;
  p.cols = cols;
  p.ldx = ldx;
  p.ldq = ldq;
  const int64_t col_groups = ceil_div(padded / 128, (int64_t)kActBlocks);
  p.col_groups = static_cast<int32_t>(col_groups);
  const float eps32 = 1e-12f;
  uint32_t bits;
  memcpy(&bits, &eps32, 4);
  bits = (bits + 0x7FFFu + ((bits >> 16) & 1u)) & 0xFFFF0000u;
  float eps_bf16;
  memcpy(&eps_bf16, &bits, 4);
  p.eps = eps_mode == FSH_EPS_FP32 ? eps32 : eps_bf16;
  // A launch's threads are counted in 32 bits: 2^24 - 1 workgroups.  A narrow
  // matrix of more rows than that (268 M of up to 512 columns) takes several.
  constexpr int64_t kMaxGrid = (1LL << 32) / kActThreads - 1;
  if (col_groups > kMaxGrid) return fail(FSH_ENOTSUP, "fsh_act_quant_1x128: too many tiles");
  const int64_t rows_per_launch = kMaxGrid / col_groups * kActRows;
  for (p.first_row = 0; p.first_row < rows; p.first_row += rows_per_launch) {
    const int64_t left = rows - p.first_row, now = left < rows_per_launch ? left : rows_per_launch;
    hipLaunchKernelGGL(act_quant_1x128_kernel, dim3(static_cast<uint32_t>(ceil_div(now, (int64_t)kActRows) * col_groups)),
                       dim3(kActThreads), 0, static_cast<hipStream_t>(stream), p);
    if (int rc = check_launch("act_quant_1x128_kernel")) return rc;
  }
  return FSH_OK;
}

namespace fsh {
namespace {

// Which tiles a product takes: the ones with the lowest estimated time.
// Measured (us with 64 x 64 tiles of three stages, 128 x 128 of two, 256 x 256;
// weights in the last-level cache; block scales, the
// column-scale variant runs 5-10 % longer on all three):
//   48 x 14336, k 4096     14.5   24.9   35.5      48 x 4096, k 14336  34.6  69.8  112
//   256 x 4096, k 4096     13.0   23.4   27.6      1000 x 2048, k 5120 22.1  31.4  46.3
//   1024 x 4096, k 4096    30.7   26.9   38.3      2048 x 4096, k 4096 55.1  39.4  42.0
//   1024 x 14336, k 4096   95.6   71.4   54.3      4096 x 4096, k 4096 112   73.0  58.8
//
// A compute unit with one workgroup to run has LDS to spare: more stages,
// i.e. more operand requests in flight ("deep").  Not where a unit runs several, whose
// requests cover one another's waits (us, fewer / more stages, weights from memory):
//   64 x 64, 3 / 4 stages:    48 x 14336, k 4096 18.6 / 16.2   48 x 4096, k 14336 48.2 / 36.1
//                             512 x 4096, k 4096 17.6 / 18.4 (column scales 20.6 / 19.2)   1024 x 4096, k 4096 32.5 / 32.6
//   128 x 128, 2 / 4 stages:  1024 x 4096, k 8192 55.9 / 46.9   1000 x 2048, k 5120 30.8 / 29.6   1000 x 5120, k 2048 20.3 / 28.3
// (eight stages of 64 x 64 tiles: 18.2 and 35.7 us on the first two, 0.4 us more where k is short)
enum Fp8TileKind {
  kFp8Tiles64 = FSH_TILES_64,
  kFp8Tiles64Deep = FSH_TILES_64_DEEP,
  kFp8Tiles128 = FSH_TILES_128,
  kFp8Tiles128Deep = FSH_TILES_128_DEEP,
  kFp8Tiles256 = FSH_TILES_256,
  kFp8Tiles256LongK = FSH_TILES_256_LONG_K,
};
Fp8TileKind fp8_tile_kind(int64_t m, int64_t n, int64_t k, bool column_scales, int64_t units) {
  static constexpr TileShape kShapes[] = {
      {64, 64, 768.0, 0.22, 0.34, 0.61, 2.0},    // three workgroups per compute unit
      {128, 128, 512.0, 0.56, 0.69, 1.07, 4.0},  // two
      {256, 256, 256.0, 0.72, 0.99, 1.48, 5.0},  // one; a round of at most half as many is cut into half tiles
  };
  const double ktiles = static_cast<double>(k / 128);
  int best = 0;
  double best_us = 0.0;
  int64_t best_tiles = 0;
  for (int i = 0; i < 3; ++i) {
    const int64_t tiles = ceil_div(m, kShapes[i].m) * ceil_div(n, kShapes[i].n);
    const double us = rounds_us(kShapes[i], static_cast<double>(tiles), static_cast<double>(tiles) * ktiles, ktiles);
    if (i == 0 || us < best_us) {
      best = i;
      best_us = us;
      best_tiles = tiles;
    }
  }
  if (best == 0) return best_tiles <= (column_scales ? 2 * units : units) ? kFp8Tiles64Deep : kFp8Tiles64;
  if (best == 1) return best_tiles <= units ? kFp8Tiles128Deep : kFp8Tiles128;
  // (One kernel; the name tells contractions of more than 256 k-tiles apart.)
  return !column_scales && k / 128 > 256 ? kFp8Tiles256LongK : kFp8Tiles256;
}

template <typename Cfg, int kBlocksPerUnit>
int launch_fp8_tiles(Fp8GemmParams& p, bool column_scales, hipStream_t stream) {
  GemmParams& s = p.schedule;
  s.tiles_m = static_cast<int32_t>(ceil_div(p.m, static_cast<int64_t>(Cfg::BM)));
  s.tiles_n = static_cast<int32_t>(ceil_div(p.n, static_cast<int64_t>(Cfg::BN)));
  const int64_t tiles = static_cast<int64_t>(s.tiles_m) * s.tiles_n;
  s.tiles_per_matrix = static_cast<int32_t>(tiles);  // (few: the rule above prefers large tiles from a few thousand on)
  s.work_items = tiles;
  s.items_per_xcd = ceil_div(tiles, static_cast<int64_t>(kXcds));
  const dim3 grid(static_cast<uint32_t>(s.items_per_xcd * kXcds)), block(Cfg::kThreads);
  static LdsReservation reserved_block_scales, reserved_column_scales;
  if (column_scales) {
    if (int rc = reserve_lds_once(reserved_column_scales, &fp8_gemm_tiles_kernel<Cfg, true, kBlocksPerUnit>, Cfg::kLdsBytes)) return rc;
    hipLaunchKernelGGL((fp8_gemm_tiles_kernel<Cfg, true, kBlocksPerUnit>), grid, block, Cfg::kLdsBytes, stream, p);
  } else {
    if (int rc = reserve_lds_once(reserved_block_scales, &fp8_gemm_tiles_kernel<Cfg, false, kBlocksPerUnit>, Cfg::kLdsBytes)) return rc;
    hipLaunchKernelGGL((fp8_gemm_tiles_kernel<Cfg, false, kBlocksPerUnit>), grid, block, Cfg::kLdsBytes, stream, p);
  }
  return check_launch("fp8_gemm_tiles_kernel");
}

// Shared checks and launch of the FP8 GEMM variants.  `p` arrives with
// the operands, sizes and scale tables filled in.
int launch_fp8_gemm(Fp8GemmParams& p, bool column_scales, const char* who, void* stream) {
  if (p.m < 0 || p.n < 0 || p.k < 0) return fail(FSH_EINVAL, "%s: negative size", who);
  if (p.m == 0 || p.n == 0) return FSH_OK;
  if (!p.xq || !p.xs || !p.wq || !p.out || (column_scales ? !p.cs : !p.ws)) return fail(FSH_EINVAL, "%s: null pointer", who);
  if (p.k == 0 || p.k % 128)
    return fail(FSH_ENOTSUP, "%s: k must be a positive multiple of 128 (pad the operands), got %lld", who, (long long)p.k);
  if (p.k >= (1LL << 31)) return fail(FSH_ENOTSUP, "%s: k must be below 2^31, got %lld", who, (long long)p.k);
  if (!column_scales && (p.k / 128) * p.ws_kb * 4 >= (1LL << 31))
    return fail(FSH_ENOTSUP, "%s: a row of the weight scale table spans more than 2 GiB", who);
  if (p.ldxq < p.k || p.ldwq < p.k || p.ldo < p.n)
    return fail(FSH_EINVAL, "%s: a leading dimension is smaller than its row", who);
  if (p.ldxq % 16 || p.ldwq % 16 || !aligned(p.xq, 16) || !aligned(p.wq, 16) || !aligned(p.out, 2))
    return fail(FSH_ENOTSUP, "%s: operand rows must be 16-byte aligned", who);
  if (static_cast<int64_t>(Fp8Gemm::BN) * p.ldwq >= (1LL << 31) || static_cast<int64_t>(Fp8Gemm::BM) * p.ldxq >= (1LL << 31) ||
      p.m >= (1LL << 29) || p.n >= (1LL << 29))
    return fail(FSH_ENOTSUP, "%s: a tile spans more than 2 GiB", who);
  GemmParams& s = p.schedule;
  memset(&s, 0, sizeof(s));
#ifdef FSH_TRACE
  if (const char* e = getenv("FSH_GEMM_TRACE")) s.trace = reinterpret_cast<uint64_t*>(strtoull(e, nullptr, 0));
#endif
  s.tiles_m = static_cast<int32_t>(ceil_div(p.m, (int64_t)Fp8Gemm::BM));
  s.tiles_n = static_cast<int32_t>(ceil_div(p.n, (int64_t)Fp8Gemm::BN));
  const int64_t tiles = static_cast<int64_t>(s.tiles_m) * s.tiles_n;
  if (tiles > 0x3FFFFFFFLL) return fail(FSH_ENOTSUP, "%s: too many tiles", who);
  s.tiles_per_matrix = static_cast<int32_t>(tiles);
  const int64_t units = compute_units();
  const hipStream_t on = static_cast<hipStream_t>(stream);
  const Fp8TileKind kind = fp8_tile_kind(p.m, p.n, p.k, column_scales, units);
  switch (kind) {
    case kFp8Tiles64: return launch_fp8_tiles<Fp8Tiles<2, 2, 1, 1, 3>, 3>(p, column_scales, on);
    case kFp8Tiles64Deep: return launch_fp8_tiles<Fp8Tiles<2, 2, 1, 1, 4>, 2>(p, column_scales, on);
    case kFp8Tiles128: return launch_fp8_tiles<Fp8Tiles<2, 2, 2, 2, 2>, 2>(p, column_scales, on);
    case kFp8Tiles128Deep: return launch_fp8_tiles<Fp8Tiles<2, 2, 2, 2, 4>, 1>(p, column_scales, on);
    default: break;
  }
  // A workgroup holds a CU for a tile, so the tiles go through the chip in
  // rounds of one per CU.  A last round that is at most half full is cut into
  // half tiles, twice as many workgroups of half the length: e.g. the 896
  // tiles of a [14336, 4096] result take 3.5 rounds instead of 4.
  const int64_t tail = units > 0 ? tiles % units : 0;
  const int64_t cut = (tail > 0 && 2 * tail <= units) ? tail : 0;
  s.work_items = tiles - cut;
  s.items_per_xcd = ceil_div(s.work_items, static_cast<int64_t>(kXcds));
  p.whole_grid = s.items_per_xcd * kXcds;
  p.half_items = 2 * cut;
  p.half_items_per_xcd = ceil_div(p.half_items, static_cast<int64_t>(kXcds));
  static LdsReservation reserved_block_scales, reserved_column_scales;
  if (int rc = column_scales ? reserve_lds_once(reserved_column_scales, &fp8_gemm_blockwise_kernel<true>, Fp8Gemm::kLdsBytes)
                             : reserve_lds_once(reserved_block_scales, &fp8_gemm_blockwise_kernel<false>, Fp8Gemm::kLdsBytes))
    return rc;
  const dim3 grid(static_cast<uint32_t>(p.whole_grid + p.half_items_per_xcd * kXcds)), block(Fp8Gemm::kThreads);
  if (column_scales)
    hipLaunchKernelGGL(fp8_gemm_blockwise_kernel<true>, grid, block, Fp8Gemm::kLdsBytes, on, p);
  else
    hipLaunchKernelGGL(fp8_gemm_blockwise_kernel<false>, grid, block, Fp8Gemm::kLdsBytes, on, p);
  return check_launch("fp8_gemm_blockwise_kernel");
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_fp8_gemm_tiles(int64_t m, int64_t n, int64_t k, int32_t column_scales) {
  using namespace fsh;
  if (m <= 0 || n <= 0 || k <= 0 || k % 128) return fail(FSH_EINVAL, "fsh_fp8_gemm_tiles: bad sizes");
  const int64_t units = compute_units();
  return fp8_tile_kind(m, n, k, column_scales != 0, units > 0 ? units : kXcds * 32);
}

FSH_API int fsh_fp8_gemm_1x128_128x128_bias(const void* xq_dev, const float* xs_dev, const void* wq_dev,
                                            const float* ws_dev, const void* bias_dev, void* out_dev, int64_t m,
                                            int64_t n, int64_t k, int64_t ldxq, int64_t ldwq, int64_t ldo,
                                            int64_t ws_cols, void* stream) {
  using namespace fsh;
  if (k > 0 && ws_cols < k / 128)
    return fail(FSH_EINVAL, "fsh_fp8_gemm_1x128_128x128: the weight scale table has %lld columns, k / 128 = %lld",
                (long long)ws_cols, (long long)(k / 128));
  if (!aligned(bias_dev, 2)) return fail(FSH_ENOTSUP, "fsh_fp8_gemm_1x128_128x128: the bias must be 2-byte aligned");
  Fp8GemmParams p;
  memset(&p, 0, sizeof(p));
  p.xq = static_cast<const uint8_t*>(xq_dev);
  p.xs = xs_dev;
  p.wq = static_cast<const uint8_t*>(wq_dev);
  p.ws = ws_dev;
  p.out = static_cast<uint16_t*>(out_dev);
  p.bias = static_cast<const uint16_t*>(bias_dev);
  p.m = m; p.n = n; p.k = k;
  p.ldxq = ldxq; p.ldwq = ldwq; p.ldo = ldo;
  p.ws_cb = ws_cols; p.ws_kb = 1;
  return launch_fp8_gemm(p, false, "fsh_fp8_gemm_1x128_128x128", stream);
}

FSH_API int fsh_fp8_gemm_1x128_128x128(const void* xq_dev, const float* xs_dev, const void* wq_dev,
                                       const float* ws_dev, void* out_dev, int64_t m, int64_t n, int64_t k,
                                       int64_t ldxq, int64_t ldwq, int64_t ldo, int64_t ws_cols, void* stream) {
  return fsh_fp8_gemm_1x128_128x128_bias(xq_dev, xs_dev, wq_dev, ws_dev, nullptr, out_dev, m, n, k, ldxq, ldwq, ldo,
                                         ws_cols, stream);
}

FSH_API int fsh_fp8_gemm_1x128_128x128_dgrad(const void* gq_dev, const float* gs_dev, const void* wtq_dev,
                                             const float* ws_dev, void* out_dev, int64_t m, int64_t in_dim,
                                             int64_t out_dim, int64_t ldgq, int64_t ldwt, int64_t ldo,
                                             int64_t ws_cols, void* stream) {
  using namespace fsh;
  if (in_dim > 0 && ws_cols < ceil_div(in_dim, (int64_t)128))
    return fail(FSH_EINVAL, "fsh_fp8_gemm_1x128_128x128_dgrad: the weight scale table has %lld columns, in_dim needs %lld",
                (long long)ws_cols, (long long)ceil_div(in_dim, (int64_t)128));
  Fp8GemmParams p;
  memset(&p, 0, sizeof(p));
  p.xq = static_cast<const uint8_t*>(gq_dev);
  p.xs = gs_dev;
  p.wq = static_cast<const uint8_t*>(wtq_dev);
  p.ws = ws_dev;
  p.out = static_cast<uint16_t*>(out_dev);
  p.m = m; p.n = in_dim; p.k = out_dim;
  p.ldxq = ldgq; p.ldwq = ldwt; p.ldo = ldo;
  p.ws_cb = 1; p.ws_kb = ws_cols;  // the weight's table read across: (input block, output block)
  return launch_fp8_gemm(p, false, "fsh_fp8_gemm_1x128_128x128_dgrad", stream);
}

FSH_API int fsh_fp8_gemm_1x128_128x1(const void* aq_dev, const float* as_dev, const void* bq_dev,
                                     const float* bs_dev, void* out_dev, int64_t m, int64_t n, int64_t k,
                                     int64_t ldaq, int64_t ldbq, int64_t ldo, void* stream) {
  using namespace fsh;
  Fp8GemmParams p;
  memset(&p, 0, sizeof(p));
  p.xq = static_cast<const uint8_t*>(aq_dev);
  p.xs = as_dev;
  p.wq = static_cast<const uint8_t*>(bq_dev);
  p.cs = bs_dev;
  p.out = static_cast<uint16_t*>(out_dev);
  p.m = m; p.n = n; p.k = k;
  p.ldxq = ldaq; p.ldwq = ldbq; p.ldo = ldo;
  return launch_fp8_gemm(p, true, "fsh_fp8_gemm_1x128_128x1", stream);
}
