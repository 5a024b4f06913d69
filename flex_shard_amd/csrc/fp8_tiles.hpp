// The scaled FP8 product on small tiles: few tokens, few columns, anything
// that does not fill the chip with the 256 x 256 tiles of fp8_linear.hip.
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

// acc[n] += (product[n] * row_scale) * (column_scales of lane n of this lane's row of 16).
// The broadcast is the multiply-add's own operand modifier (the compiler keeps
// a separate move per element when given the builtin).  column_scales comes
// from LDS, not from the vector ALU, so the modifier's read needs no wait states.
template <int N = 0>
__device__ __forceinline__ void fold_with_row_broadcast(f32x16& acc, const f32x16& product, float row_scale,
                                                        float column_scales) {
  if constexpr (N < 16) {
    const float scaled = product[N] * row_scale;
    float sum = acc[N];
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(sum)
        : "v"(column_scales), "v"(scaled), "n"(N));
    acc[N] = sum;
    fold_with_row_broadcast<N + 1>(acc, product, row_scale, column_scales);
  }
}

// The same for a block of 16 x 16: element r takes the scale of lane 4 block + r
// of its row of 16 lanes (block is a constant after unrolling).
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

// Four waves, WM x WN, each TM x TN blocks of 32 x 32; a k-tile is one scale
// block (128 bytes of every row) with its row scales and column scales.
template <int WM_, int WN_, int TM_, int TN_, int kStages_>
struct Fp8Tiles {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, kStages = kStages_;
  static constexpr int kWaveM = 32 * TM, kWaveN = 32 * TN, BM = WM * kWaveM, BN = WN * kWaveN, BK = 128;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves, kRowBytes = 128;
  static constexpr int kABytes = BM * kRowBytes, kScaleOffset = (BM + BN) * kRowBytes;
  static constexpr int kStageBytes = kScaleOffset + (BM + BN) * 4;
  static constexpr int kFillRows = 8 * kWaves;
  static constexpr int kLoadsA = BM / kFillRows, kLoadsB = BN / kFillRows;
  static constexpr int kRequests = kLoadsA + kLoadsB + 1;     // per wave and k-tile; the last one brings 64 scales
  static constexpr int kScaleRequests = (BM + BN) / 64;       // per workgroup: waves past them repeat
  static constexpr int kPitch = kWaveN * 2 + 8, kRegion = kWaveM * kPitch;
  static constexpr int kLdsBytes = kStages * kStageBytes;
  static_assert(BN <= 128, "a tile's columns share one block scale");
  static_assert(BM % 64 == 0 && BN % 64 == 0 && kWaves % kScaleRequests == 0, "scale requests of 64");
  static_assert(kWaves * kRegion <= kLdsBytes, "the images fit the loop's LDS");
};

template <typename Cfg, bool kColumnScales, int kBlocksPerUnit>
__global__ __launch_bounds__(Cfg::kThreads, kBlocksPerUnit * Cfg::kWaves / 4) void fp8_gemm_tiles_kernel(const Fp8GemmParams p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  constexpr int TM = Cfg::TM, TN = Cfg::TN, kStages = Cfg::kStages, kBlocks = TM * TN;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  int64_t unused_batch;
  int tm, tn;
  if (!tile_of_workgroup(p.schedule, blockIdx.x, &unused_batch, &tm, &tn)) return;  // whole workgroup
  const int64_t m0 = static_cast<int64_t>(uniform_i32(tm)) * Cfg::BM, n0 = static_cast<int64_t>(uniform_i32(tn)) * Cfg::BN;
  const int ktiles = static_cast<int>(p.k / Cfg::BK);

  // Load side, as in the bf16 tile kernel; rows past the matrix are read from
  // its last row (their products are never stored).
  const int fill_row = 8 * wave + (lane >> 3);
  const int fill_chunk = (lane & 7) ^ ((fill_row >> 1) & 7);
  const uint8_t* src[Cfg::kLoadsA + Cfg::kLoadsB];
#pragma unroll
  for (int q = 0; q < Cfg::kLoadsA; ++q) {
    const int64_t r = m0 + Cfg::kFillRows * q + fill_row;
    src[q] = p.xq + (r < p.m ? r : p.m - 1) * p.ldxq + fill_chunk * 16;
  }
#pragma unroll
  for (int q = 0; q < Cfg::kLoadsB; ++q) {
    const int64_t r = n0 + Cfg::kFillRows * q + fill_row;
    src[Cfg::kLoadsA + q] = p.wq + (r < p.n ? r : p.n - 1) * p.ldwq + fill_chunk * 16;
  }
  // The wave's scale request: 64 row scales, or 64 column scales -- the block
  // scale 64 times in the block-scale variant.
  const int scale_request = wave % Cfg::kScaleRequests;
  const bool scales_rows = scale_request < Cfg::BM / 64;
  const int64_t scale_at = (scales_rows ? m0 + 64 * scale_request : n0 + 64 * (scale_request - Cfg::BM / 64)) + lane;
  const float* scale_src;
  int64_t scale_step;
  if (scales_rows) {
    scale_src = p.xs + (scale_at < p.m ? scale_at : p.m - 1);
    scale_step = p.m;
  } else if (kColumnScales) {
    scale_src = p.cs + (scale_at < p.n ? scale_at : p.n - 1);
    scale_step = p.n;
  } else {
    scale_src = p.ws + n0 / 128 * p.ws_cb;
    scale_step = p.ws_kb;
  }
  typedef __attribute__((address_space(3))) uint8_t* lds_address;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_address)lds_bytes));
  auto request = [&](int kt, uint32_t stage, int idx) {
    const uint32_t at = lds_base + stage * Cfg::kStageBytes;
    if (idx < Cfg::kLoadsA + Cfg::kLoadsB)  // (operand B's rows follow operand A's in the stage)
      dma_load_16_at(src[idx] + static_cast<int64_t>(kt) * Cfg::kRowBytes,
                     at + wave * 1024 + idx * (Cfg::kFillRows * Cfg::kRowBytes));
    else
      dma_load_4_at(reinterpret_cast<const uint8_t*>(scale_src + kt * scale_step), at + Cfg::kScaleOffset + scale_request * 256);
  };

  // Fragment side: row = lane & 31 of a 32-row block; chunks 4 kh + 2 h and
  // 4 kh + 2 h + 1 of the row (kh = 64-byte half), each in slot chunk ^ ((row >> 1) & 7).
  const int frag_row = lane & 31, h = lane >> 5;
  uint32_t frag_off[2][2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      frag_off[kh][c] = static_cast<uint32_t>(frag_row * Cfg::kRowBytes + (((4 * kh + 2 * h + c) ^ ((frag_row >> 1) & 7)) * 16));
  auto read_frag = [&](const uint8_t* block, v8i32 (&frag)[2]) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(block + frag_off[kh][0]);
      const u32x4 hi = *reinterpret_cast<const u32x4*>(block + frag_off[kh][1]);
      frag[kh] = v8i32{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z), static_cast<int>(lo.w),
                       static_cast<int>(hi.x), static_cast<int>(hi.y), static_cast<int>(hi.z), static_cast<int>(hi.w)};
    }
  };
  constexpr int kSets = kBlocks == 1 ? 2 : 1;  // a lone block reads the next k-tile's fragments while it multiplies
  v8i32 afrag[kSets][TM][2], bfrag[kSets][TN][2];
  auto read_a = [&](uint32_t stage, int set, int i) {
    read_frag(lds_bytes + stage * Cfg::kStageBytes + (wm * Cfg::kWaveM + i * 32) * Cfg::kRowBytes, afrag[set][i]);
  };
  auto read_b = [&](uint32_t stage, int set, int j) {
    read_frag(lds_bytes + stage * Cfg::kStageBytes + Cfg::kABytes + (wn * Cfg::kWaveN + j * 32) * Cfg::kRowBytes, bfrag[set][j]);
  };
  // Row scales of the wave's rows, times the block scale in the block-scale
  // variant; per-column scales arranged for fold_with_row_broadcast: in every
  // row of 16 lanes, lane n holds the scale of accumulator element n.
  float row_scale[TM], col_scale[TN];
  auto read_scales = [&](uint32_t stage) {
    const float* rows = reinterpret_cast<const float*>(lds_bytes + stage * Cfg::kStageBytes + Cfg::kScaleOffset);
    const float* cols = rows + Cfg::BM;
#pragma unroll
    for (int i = 0; i < TM; ++i) row_scale[i] = rows[wm * Cfg::kWaveM + i * 32 + frag_row];
    if (kColumnScales) {
#pragma unroll
      for (int j = 0; j < TN; ++j) col_scale[j] = cols[wn * Cfg::kWaveN + j * 32 + 8 * ((lane & 15) >> 2) + 4 * h + (lane & 3)];
    } else {
      const float block_scale = cols[0];
#pragma unroll
      for (int i = 0; i < TM; ++i) row_scale[i] *= block_scale;
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  auto multiply = [&](int set, int i, int j) -> f32x16 {
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const f32x16 half = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bfrag[set][j][0], afrag[set][i][0], zero, 0, 0, 0, 0, 0, 0);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bfrag[set][j][1], afrag[set][i][1], half, 0, 0, 0, 0, 0, 0);
  };
  auto fold = [&](const f32x16& product, int i, int j) {
    if (kColumnScales) {
      fold_with_row_broadcast(acc[i][j], product, row_scale[i], col_scale[j]);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(product[r], row_scale[i], acc[i][j][r]);
    }
  };
  // This wave's part of the k-tile after `kt` has landed (those behind it stay
  // in flight), everyone's has behind the barrier, and everyone holds in
  // registers what it still needs of kt's own stage.
  auto hand_over = [&](int kt) {
    const int behind = ktiles - 2 - kt;
    if (kStages >= 4 && behind >= kStages - 2)
      wait_for_dma_loads_but<(kStages - 2) * Cfg::kRequests>();
    else if (kStages >= 4 && behind >= (kStages - 2) / 2)
      wait_for_dma_loads_but<(kStages - 2) / 2 * Cfg::kRequests>();
    else if (kStages == 3 && behind >= 1)
      wait_for_dma_loads_but<Cfg::kRequests>();
    else
      wait_for_dma_loads();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

#pragma unroll
  for (int kt = 0; kt < kStages; ++kt)
    if (kt < ktiles) {
#pragma unroll
      for (int idx = 0; idx < Cfg::kRequests; ++idx) request(kt, kt, idx);
    }
  hand_over(-1);
  read_a(0, 0, 0);
  read_b(0, 0, 0);
  uint32_t stage = 0;
  // One k-tile; `more`: kt + 1 exists, `ahead`: kt + kStages does.
  auto k_tile = [&](int kt, auto set_tag, auto more_tag, auto ahead_tag) {
    constexpr int set = decltype(set_tag)::value;
    constexpr bool more = decltype(more_tag)::value, ahead = decltype(ahead_tag)::value;
    const uint32_t after = stage + 1 == kStages ? 0 : stage + 1;
    read_scales(stage);
    if constexpr (kBlocks == 1) {
      if (more) {
        hand_over(kt);
        read_a(after, set ^ 1, 0);
        read_b(after, set ^ 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      const f32x16 product = multiply(set, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (ahead) {
#pragma unroll
        for (int idx = 0; idx < Cfg::kRequests; ++idx) request(kt + kStages, stage, idx);
      }
      fold(product, 0, 0);
    } else {
      // The blocks in the order (0,0) (1,0) (0,1) (1,1): the first one's
      // fragments are free at the last, whose MFMAs cover the read of the next
      // k-tile's first ones; a block is folded behind the next one's MFMAs.
      static_assert(kBlocks == 1 || (TM == 2 && TN == 2), "block order");
      f32x16 part[2];
      read_a(stage, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
      part[0] = multiply(0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      read_b(stage, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
      part[1] = multiply(0, 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      fold(part[0], 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      part[0] = multiply(0, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
      fold(part[1], 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        hand_over(kt);
        read_a(after, 0, 0);
        read_b(after, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      part[1] = multiply(0, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      if (ahead) {
#pragma unroll
        for (int idx = 0; idx < Cfg::kRequests; ++idx) request(kt + kStages, stage, idx);
      }
      fold(part[0], 0, 1);
      fold(part[1], 1, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    stage = after;
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, kSets - 1> odd{};
  int kt = 0;
  for (; kt + 1 + kStages < ktiles; kt += 2) {
    k_tile(kt, even, yes, yes);
    k_tile(kt + 1, odd, yes, yes);
  }
  for (; kt < ktiles; ++kt) {  // the last few, fragments back in set 0 after each pair
    const bool more = kt + 1 < ktiles, ahead = kt + kStages < ktiles;
    if (kSets == 1 || (kt & 1) == 0) {
      if (ahead) k_tile(kt, even, yes, yes);
      else if (more) k_tile(kt, even, yes, no);
      else k_tile(kt, even, no, no);
    } else {
      if (ahead) k_tile(kt, odd, yes, yes);
      else if (more) k_tile(kt, odd, yes, no);
      else k_tile(kt, odd, no, no);
    }
  }
  __syncthreads();  // the images overlay the stages

  uint8_t* region = lds_bytes + wave * Cfg::kRegion;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *reinterpret_cast<u32x2*>(region + (i * 32 + frag_row) * Cfg::kPitch + (j * 32 + 8 * b + 4 * h) * 2) =
            u32x2{pack_bf16x2(acc[i][j][4 * b], acc[i][j][4 * b + 1]),
                  pack_bf16x2(acc[i][j][4 * b + 2], acc[i][j][4 * b + 3])};
  wave_lds_sync();
  store_fp8_product<Cfg::kWaveM, Cfg::kWaveN, Cfg::kPitch>(region, p, m0 + wm * Cfg::kWaveM, n0 + wn * Cfg::kWaveN, lane);
}

}  // namespace
}  // namespace fsh
