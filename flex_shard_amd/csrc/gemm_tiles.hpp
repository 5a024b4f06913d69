// The bf16 NT GEMM for every problem the 256 x 256 kernel does not take: any
// M, N and K % 8 == 0, few tiles, ragged edges, several problems per launch.
#pragma once
#include "mfma_tiles.hpp"

namespace fsh {
namespace {

using TileLaunch = GemmLaunchOf<8>;

// WM x WN waves, each TM x TN blocks of 32 x 32.  kStages k-tiles of 64 in LDS.
template <int WM_, int WN_, int TM_, int TN_, int kStages_>
struct GemmTiles {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, kStages = kStages_;
  static constexpr int kWaveM = 32 * TM, kWaveN = 32 * TN, BM = WM * kWaveM, BN = WN * kWaveN, BK = 64, KS = BK / 16;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kRowBytes = BK * 2;  // 128
  static constexpr int kOperandABytes = BM * kRowBytes;
  static constexpr int kStageBytes = (BM + BN) * kRowBytes;
  // A wave-level request fills 1 KB = 8 tile rows.
  static constexpr int kFillRows = 8 * kWaves;
  static constexpr int kLoadsA = BM / kFillRows, kLoadsB = BN / kFillRows, kLoads = kLoadsA + kLoadsB;
  // k steps whose fragments are read ahead of their MFMAs: enough MFMAs have
  // to issue under an LDS read to cover it.
  static constexpr int kAhead = TM * TN >= 4 ? 1 : 3, kSets = TM * TN >= 4 ? 2 : 4;
  // Epilogue: one [kWaveM][kWaveN] bf16 image per wave, rows 8 bytes off a
  // multiple of the bank window.
  static constexpr int kPitch = kWaveN * 2 + 8;   // [row][col]
  static constexpr int kPitchT = kWaveM * 2 + 8;  // [col][row]
  static constexpr int kRegion = max_int(kWaveM * kPitch, kWaveN * kPitchT);
  static constexpr int kLdsBytes = kStages * kStageBytes;
  static_assert(kWaves * kRegion <= kLdsBytes, "the images fit the loop's LDS");
  static_assert(BM % kFillRows == 0 && BN % kFillRows == 0, "whole requests");
};

// Finals bf16(fma(beta, D, alpha * acc) + diagonal term) of a wave's sub-tile
// at (row0, col0), through its LDS image: D arrives row-wise, C and the
// transposed (or mirrored) output leave row-wise.  Only the wave itself
// touches its image, so program order is all the synchronization there is.
template <typename Cfg>
__device__ __forceinline__ void store_wave_tile(const GemmParams& p, int64_t batch, int64_t row0, int64_t col0, int lane,
                                                bool mirror, f32x16 (&acc)[Cfg::TM][Cfg::TN], uint8_t* region) {
  constexpr int TM = Cfg::TM, TN = Cfg::TN;
  uint16_t* C = p.C + batch * p.sC;
  uint16_t* Ct = mirror ? C : (p.Ct ? p.Ct + batch * p.sCt : nullptr);
  const int64_t ldct = mirror ? p.ldc : p.ldct;
  const int r_lane = lane & 31, h = lane >> 5;
  auto slot = [&](int i, int j, int b) -> u32x2* {  // accumulators 4 b .. 4 b + 3 of block (i, j)
    return reinterpret_cast<u32x2*>(region + (i * 32 + r_lane) * Cfg::kPitch + (j * 32 + 8 * b + 4 * h) * 2);
  };

  const bool has_d = p.D != nullptr;
  u32x2 dv[TM][TN][4];
  if (has_d) {
    constexpr int kLanesPerRow = Cfg::kWaveN / 8, kRowsPerPass = 64 / kLanesPerRow, kPasses = Cfg::kWaveM / kRowsPerPass;
    const uint16_t* D = p.D + batch * p.sD;
    const bool vec = rows_are_16_byte(D, p.ldd);
    const int r0 = lane / kLanesPerRow, chunk = lane % kLanesPerRow;
    const int64_t col = col0 + chunk * 8;
    u32x4 t[kPasses];
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
      const int64_t row = row0 + pass * kRowsPerPass + r0;
      t[pass] = u32x4{0, 0, 0, 0};
      if (row < p.M && col < p.N) t[pass] = load_row_piece(D + row * p.ldd, col, p.N, vec);
    }
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
      uint8_t* d = region + (pass * kRowsPerPass + r0) * Cfg::kPitch + chunk * 16;
      *reinterpret_cast<u32x2*>(d) = u32x2{t[pass].x, t[pass].y};
      *reinterpret_cast<u32x2*>(d + 8) = u32x2{t[pass].z, t[pass].w};
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int b = 0; b < 4; ++b) dv[i][j][b] = *slot(i, j, b);
  }
  u32x2 fin[TM][TN][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = p.alpha * acc[i][j][4 * b + t];  // alpha == 1 is exact
        if (has_d) {
          v[0] = __builtin_fmaf(p.beta, u32_as_f32(dv[i][j][b].x << 16), v[0]);
          v[1] = __builtin_fmaf(p.beta, u32_as_f32(dv[i][j][b].x & 0xFFFF0000u), v[1]);
          v[2] = __builtin_fmaf(p.beta, u32_as_f32(dv[i][j][b].y << 16), v[2]);
          v[3] = __builtin_fmaf(p.beta, u32_as_f32(dv[i][j][b].y & 0xFFFF0000u), v[3]);
        }
        if (p.diag_add != 0.0f && row0 + 32 * i == col0 + 32 * j) {  // (sub-tiles start at multiples of 32)
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = r_lane == 8 * b + 4 * h + t ? v[t] + p.diag_add : v[t];
        }
        fin[i][j][b] = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b) *slot(i, j, b) = fin[i][j][b];
  wave_lds_sync();
  store_wave_image<Cfg::kWaveM, Cfg::kWaveN, Cfg::kPitch>(region, C, p.ldc, row0, col0, p.M, p.N, lane);
  if (Ct == nullptr) return;  // uniform over the workgroup
  wave_lds_sync();  // the row reads are done before the image is written again as [col][row]
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t pair = (t >> 1) ? fin[i][j][b].y : fin[i][j][b].x;
          *reinterpret_cast<uint16_t*>(region + (j * 32 + 8 * b + 4 * h + t) * Cfg::kPitchT + (i * 32 + r_lane) * 2) =
              static_cast<uint16_t>((t & 1) ? (pair >> 16) : pair);
        }
  wave_lds_sync();
  store_wave_image<Cfg::kWaveN, Cfg::kWaveM, Cfg::kPitchT>(region, Ct, ldct, col0, row0, p.N, p.M, lane);
}

// What bounds it: the request path of a compute unit takes a 1 KB request per
// 16 cycles, so the 32 requests of a 128 x 128 x 64 k-tile last as long as its
// MFMAs (512 cycles), and a request holds up the wave that issues it; each is
// therefore issued behind an MFMA, fragments are read a k step ahead (three
// for 32 x 32 waves), and workgroups that share a compute unit cover each
// other's barriers.  6592^3 with 128 x 128 tiles: 843 TFLOP/s with the requests
// in one go at the top of a k-tile and the fragment reads behind the barrier,
// 988 rotated as below, 1054 with the loop split so that no request sits
// behind a branch of its own, 1130 with 256 x 128 tiles of eight waves.
// Against the kernels this one replaced (register-staged 128 x 128 x 32, and
// 256 x 256 x 64 with predicated accesses for ragged shapes): 6592^3 690 ->
// 532 us, 768 x 768 x 3072 (batch 4, symmetric) 45 -> 19 us, one 304 x 304 x
// 704 product 17.7 -> 5.7 us.
//
// Operands travel global -> LDS directly into swizzled 128-byte rows, as in
// the 256 x 256 kernel.  Rows past the matrix are read from its last row and
// the last k-tile's chunks past K from the row's last chunk; what they
// multiply is never stored, respectively zeroed in the fragments.
template <typename Cfg, int kBlocksPerUnit>
__global__ __launch_bounds__(Cfg::kThreads, kBlocksPerUnit * Cfg::kWaves / 4) void gemm_nt_tiles_kernel(const TileLaunch launch) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  constexpr int TM = Cfg::TM, TN = Cfg::TN, KS = Cfg::KS, kStages = Cfg::kStages, kMfmas = TM * TN, kSets = Cfg::kSets;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;

  int which = 0;
#pragma unroll
  for (int i = 1; i < TileLaunch::kMaxProblems; ++i) which += static_cast<int>(blockIdx.x) >= launch.first_workgroup[i] ? 1 : 0;
  which = uniform_i32(which);
  const GemmParams& p = launch.problem[which];
  int64_t batch;
  int tm, tn;
  if (!tile_of_workgroup(p, static_cast<int64_t>(blockIdx.x) - launch.first_workgroup[which], &batch, &tm, &tn)) return;  // whole workgroup
  batch = uniform_i64(batch);
  tm = uniform_i32(tm);
  tn = uniform_i32(tn);
  const int64_t m0 = static_cast<int64_t>(tm) * Cfg::BM, n0 = static_cast<int64_t>(tn) * Cfg::BN;

  // Load side: wave-level request q of an operand fills tile rows
  // [kFillRows q + 8 wave, +8); lane l fills slot l & 7 of row l >> 3 there.
  const int fill_row = 8 * wave + (lane >> 3);
  const int fill_chunk = (lane & 7) ^ ((fill_row >> 1) & 7);
  const uint8_t* src[Cfg::kLoads];
#pragma unroll
  for (int q = 0; q < Cfg::kLoadsA; ++q) {
    const int64_t r = m0 + Cfg::kFillRows * q + fill_row;
    src[q] = reinterpret_cast<const uint8_t*>(p.A + batch * p.sA + (r < p.M ? r : p.M - 1) * p.lda) + fill_chunk * 16;
  }
#pragma unroll
  for (int q = 0; q < Cfg::kLoadsB; ++q) {
    const int64_t r = n0 + Cfg::kFillRows * q + fill_row;
    src[Cfg::kLoadsA + q] = reinterpret_cast<const uint8_t*>(p.B + batch * p.sB + (r < p.N ? r : p.N - 1) * p.ldb) + fill_chunk * 16;
  }
  typedef __attribute__((address_space(3))) uint8_t* lds_address;
  const uint32_t fill_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_address)lds_bytes)) + wave * 1024;
  const int ktiles = static_cast<int>((p.K + Cfg::BK - 1) / Cfg::BK);
  const int tail_chunks = static_cast<int>((p.K / 8) & 7);  // 0: the last k-tile is whole
  // Byte offset of k-tile kt along the rows; chunks past K read the row's last chunk instead.
  const int64_t tail_back = tail_chunks != 0 && fill_chunk >= tail_chunks ? (fill_chunk - (tail_chunks - 1)) * 16 : 0;
  auto k_offset = [&](int kt) -> int64_t {
    return static_cast<int64_t>(kt) * Cfg::kRowBytes - (kt == ktiles - 1 ? tail_back : 0);
  };
  auto issue_one = [&](int64_t k_off, uint32_t stage, int idx) {
    // (operand B's rows follow operand A's in the stage)
    dma_load_16_at(src[idx] + k_off, fill_lds + stage * Cfg::kStageBytes + idx * (Cfg::kFillRows * Cfg::kRowBytes));
  };

  // Fragment side: lane l reads row l & 31 of a 32-row block, chunk 2 ks + (l >> 5).
  const int frag_row = lane & 31;
  const uint32_t frag_base = static_cast<uint32_t>(frag_row * Cfg::kRowBytes + (((lane >> 5) ^ ((frag_row >> 1) & 7)) * 16));
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  bf16x8 af[kSets][TM], bf[kSets][TN];
  // Fragments of k step ks of the k-tile in `stage`; `masked`: the chunks past K as zero.
  auto read_frags = [&](uint32_t stage, int ks, bool masked) {
    const uint8_t* base = lds_bytes + stage * Cfg::kStageBytes + (frag_base ^ (ks * 32));
    const uint8_t* a = base + wm * Cfg::kWaveM * Cfg::kRowBytes;
    const uint8_t* b = base + Cfg::kOperandABytes + wn * Cfg::kWaveN * Cfg::kRowBytes;
    const int set = ks % kSets;
#pragma unroll
    for (int i = 0; i < TM; ++i) af[set][i] = *reinterpret_cast<const bf16x8*>(a + i * 32 * Cfg::kRowBytes);
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[set][j] = *reinterpret_cast<const bf16x8*>(b + j * 32 * Cfg::kRowBytes);
    if (masked) {
      const bf16x8 zero = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
      const bool live = 2 * ks + (lane >> 5) < tail_chunks;
#pragma unroll
      for (int i = 0; i < TM; ++i) af[set][i] = live ? af[set][i] : zero;
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[set][j] = live ? bf[set][j] : zero;
    }
  };
  auto mfma = [&](int ks, int g) {
    const int i = g / TN, j = g % TN, set = ks % kSets;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[set][j], af[set][i], acc[i][j], 0, 0, 0);
  };
  // One k-tile, rotated by a quarter: the barrier that hands over k-tile
  // kt + 1 sits before the last k step, behind which the first fragments of
  // kt + 1 are read, and which releases kt's own stage (every wave holds its
  // last fragments in registers) to the requests for kt + kStages: half of
  // them behind the MFMAs there, half in the first k step of kt + 1.
  //   second / first: the second half of the requests for kt + kStages - 1
  //   and the first half of those for kt + kStages go out
  constexpr int kFirst = (Cfg::kLoads + 1) / 2, kSecond = Cfg::kLoads - kFirst;
  uint32_t stage = 0;  // of kt
  auto k_tile = [&](int kt, auto second_tag, auto first_tag, auto masked_tag, auto last_tag) {
    constexpr bool second = decltype(second_tag)::value, first = decltype(first_tag)::value;
    constexpr bool masked = decltype(masked_tag)::value, last = decltype(last_tag)::value;
    const uint32_t before = stage == 0 ? kStages - 1 : stage - 1, after = stage + 1 == kStages ? 0 : stage + 1;
#pragma unroll
    for (int ks = 0; ks + 1 < KS; ++ks) {
      if (ks + Cfg::kAhead < KS) read_frags(stage, ks + Cfg::kAhead, masked);
      __builtin_amdgcn_sched_barrier(0);
      const int64_t k_off = second && ks == 0 ? k_offset(kt + kStages - 1) : 0;
#pragma unroll
      for (int g = 0; g < kMfmas; ++g) {
        mfma(ks, g);
        if (second && ks == 0) {
#pragma unroll
          for (int idx = g * kSecond / kMfmas; idx < (g + 1) * kSecond / kMfmas; ++idx) issue_one(k_off, before, kFirst + idx);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!last) {
      // k-tile kt + 1 has landed (this wave's part); those behind it stay in flight.
      const int behind = ktiles - 2 - kt;
      if (kStages >= 4 && (first || behind >= 2))
        wait_for_dma_loads_but<2 * Cfg::kLoads>();
      else if (kStages >= 3 && (first || behind >= 1))
        wait_for_dma_loads_but<Cfg::kLoads>();
      else
        wait_for_dma_loads();
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < Cfg::kAhead; ++ks) read_frags(after, ks, false);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int64_t k_off = first ? k_offset(kt + kStages) : 0;
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) {
      mfma(KS - 1, g);
      if (first) {
#pragma unroll
        for (int idx = g * kFirst / kMfmas; idx < (g + 1) * kFirst / kMfmas; ++idx) issue_one(k_off, stage, idx);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    stage = after;
  };

  // Fill the pipeline: the first kStages - 1 k-tiles and half of the next.
#pragma unroll
  for (int kt = 0; kt < kStages; ++kt)
    if (kt < ktiles) {
      const int64_t k_off = k_offset(kt);
#pragma unroll
      for (int idx = 0; idx < (kt + 1 < kStages ? Cfg::kLoads : kFirst); ++idx) issue_one(k_off, kt, idx);
    }
  if (ktiles >= kStages)
    wait_for_dma_loads_but<(kStages - 2) * Cfg::kLoads + kFirst>();
  else if (kStages >= 4 && ktiles == 3)
    wait_for_dma_loads_but<2 * Cfg::kLoads>();
  else if (kStages >= 3 && ktiles == 2)
    wait_for_dma_loads_but<Cfg::kLoads>();
  else
    wait_for_dma_loads();
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int ks = 0; ks < Cfg::kAhead; ++ks) read_frags(0, ks, false);
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  int kt = 0;
  for (; kt + kStages < ktiles; ++kt) k_tile(kt, yes, yes, no, no);
  // Drain: nothing more to request but the half that is still due.
  bool due = ktiles >= kStages;
  for (; kt + 1 < ktiles; ++kt) {
    if (due) k_tile(kt, yes, no, no, no);
    else k_tile(kt, no, no, no, no);
    due = false;
  }
  if (tail_chunks != 0) {
    // the fragments read ahead were read unmasked
#pragma unroll
    for (int ks = 0; ks < Cfg::kAhead; ++ks) read_frags(stage, ks, true);
    k_tile(ktiles - 1, no, no, yes, yes);
  } else {
    k_tile(ktiles - 1, no, no, no, yes);
  }
  __syncthreads();  // the images overlay the stages
  store_wave_tile<Cfg>(p, batch, m0 + wm * Cfg::kWaveM, n0 + wn * Cfg::kWaveN, lane, p.symmetric && tn >= p.symmetric * (tm + 1), acc,
                       lds_bytes + wave * Cfg::kRegion);
}

}  // namespace
}  // namespace fsh
