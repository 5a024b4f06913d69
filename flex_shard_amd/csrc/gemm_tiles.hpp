// The bf16 NT GEMM for every problem the 256 x 256 kernel does not take: any
// M, N and K % 8 == 0, few tiles, ragged edges, several problems per launch.
#pragma once
#include "mfma_tiles.hpp"

namespace fsh {
namespace {

using TileLaunch = GemmLaunchOf<8>;

// WM x WN waves, each TM x TN blocks of 16 x 16.  Operands are requested kDepth
// k-tiles of 64 ahead: operand A has a slot for each of them and for the k-tile
// in work, operand B, which is requested later in a k-tile, for one fewer;
// kLateA: operand A as late as B, with as many slots.
template <int WM_, int WN_, int TM_, int TN_, int kDepth_, bool kLateA_ = false>
struct GemmTiles {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, kDepth = kDepth_;
  static constexpr bool kLateA = kLateA_;
  static constexpr int kWaveM = 16 * TM, kWaveN = 16 * TN, BM = WM * kWaveM, BN = WN * kWaveN, BK = 64, KS = BK / 32;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kRowBytes = BK * 2;  // 128
  static constexpr int kABytes = BM * kRowBytes, kBBytes = BN * kRowBytes;
  static constexpr int kARing = (kDepth + (kLateA ? 0 : 1)) * kABytes, kBRing = kDepth * kBBytes;  // B's ring lies behind A's
  // A wave-level request fills 1 KB = 8 tile rows.
  static constexpr int kFillRows = 8 * kWaves;
  static constexpr int kLoadsA = BM / kFillRows, kLoadsB = BN / kFillRows, kLoads = kLoadsA + kLoadsB;
  // Epilogue: one [kWaveM][kWaveN] bf16 image per wave.
  static constexpr int kPitch = kWaveN * 2 + 16, kRegion = kWaveM * kPitch;
  static constexpr int kLdsBytes = kARing + kBRing;
  static_assert(kWaves * kRegion <= kLdsBytes, "the images fit the loop's LDS");
  static_assert(BM % kFillRows == 0 && BN % kFillRows == 0 && kFillRows % 16 == 0, "whole requests");
  static_assert(kDepth >= 2 && kDepth <= 4, "the waits of the k loop's end");
};

// Finals bf16(fma(beta, D, alpha * acc) + diagonal term) of a wave's sub-tile
// at (row0, col0), through its LDS image: D arrives row-wise and C leaves
// row-wise; the transposed (or mirrored) output is read across the image, two
// transposing reads for eight rows of a column.  (Before, the image was written
// again as [col][row], 64 two-byte writes per lane of a 64 x 64 sub-tile.)
// Only the wave itself touches its image, so program order is all the
// synchronization there is.
template <typename Cfg>
__device__ __forceinline__ void store_wave_tile(const GemmParams& p, int64_t batch, int64_t row0, int64_t col0, int lane,
                                                bool mirror, f32x4 (&acc)[Cfg::TM][Cfg::TN], uint8_t* region) {
  constexpr int TM = Cfg::TM, TN = Cfg::TN;
  uint16_t* C = p.C + batch * p.sC;
  uint16_t* Ct = mirror ? C : (p.Ct ? p.Ct + batch * p.sCt : nullptr);
  const int64_t ldct = mirror ? p.ldc : p.ldct;
  const int r_lane = lane & 15, c_lane = 4 * (lane >> 4);
  auto slot = [&](int i, int j) -> u32x2* {  // the four accumulators of block (i, j)
    return reinterpret_cast<u32x2*>(region + (i * 16 + r_lane) * Cfg::kPitch + (j * 16 + c_lane) * 2);
  };

  const bool has_d = p.D != nullptr;
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
    for (int pass = 0; pass < kPasses; ++pass)
      *reinterpret_cast<u32x4*>(region + (pass * kRowsPerPass + r0) * Cfg::kPitch + chunk * 16) = t[pass];
    wave_lds_sync();
  }
  // A lane's finals replace exactly the D values it reads itself.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    u32x2 dv[TN];
    if (has_d) {
#pragma unroll
      for (int j = 0; j < TN; ++j) dv[j] = *slot(i, j);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = p.alpha * acc[i][j][t];  // alpha == 1 is exact
      if (has_d) {
        v[0] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].x << 16), v[0]);
        v[1] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].x & 0xFFFF0000u), v[1]);
        v[2] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].y << 16), v[2]);
        v[3] = __builtin_fmaf(p.beta, u32_as_f32(dv[j].y & 0xFFFF0000u), v[3]);
      }
      if (p.diag_add != 0.0f && row0 + 16 * i == col0 + 16 * j) {  // (sub-tiles start at multiples of 16)
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = r_lane == c_lane + t ? v[t] + p.diag_add : v[t];
      }
      *slot(i, j) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
  wave_lds_sync();
  store_wave_image<Cfg::kWaveM, Cfg::kWaveN, Cfg::kPitch>(region, C, p.ldc, row0, col0, p.M, p.N, lane);
  if (Ct == nullptr) return;  // uniform over the workgroup
  // Lane t of group g of 16: column t of 16, rows 8 g .. 8 g + 7 of 32.
  const bool vec = rows_are_16_byte(Ct, ldct);
  const int t = lane & 15, g = lane >> 4;
  const uint8_t* from = region + (8 * g + (t >> 2)) * Cfg::kPitch + (t & 3) * 8;
#pragma unroll
  for (int cb = 0; cb < TN; ++cb) {
    const int64_t col = col0 + cb * 16 + t;
#pragma unroll
    for (int rb = 0; rb < Cfg::kWaveM / 32; ++rb) {
      const u32x2 lo = read_lds_transposed(from + rb * 32 * Cfg::kPitch + cb * 32);
      const u32x2 hi = read_lds_transposed(from + (rb * 32 + 4) * Cfg::kPitch + cb * 32);
      const int64_t row = row0 + rb * 32 + 8 * g;
      if (col < p.N && row < p.M) store_row_piece(Ct + col * ldct, row, p.M, vec, u32x4{lo.x, lo.y, hi.x, hi.y});
    }
  }
}

// What bounds it: the request path of a compute unit takes a 1 KB request per
// 16 cycles, so the 32 requests of a 128 x 128 x 64 k-tile last as long as its
// MFMAs (512 cycles), and a request holds up the wave that issues it.  One
// 128 x 128 workgroup per compute unit takes 0.22 us per k-tile with its
// operands in LDS, 0.27 with the fragment reads or the requests and 0.30 with
// both (64 tiles; 0.40 with every compute unit busy); short contractions spend
// as long on their start and end.  16 x 16 x 32 MFMAs, a request behind every
// few of them in both k steps, scalar bases with 32-bit offsets, one orientation
// in the image, against 32 x 32 x 16 MFMAs, 64-bit addresses per request and the
// requests of a k-tile in two bunches (same bits), us:
//   2048 x 2048, k 2048 25.8 -> 20.7 (128 x 128 tiles)   4096 x 4096, k 2048 70.9 -> 58.1
//   8 x 768 x 768, 4 x 3072 x 768, 4 x 768 x 3072, ...: G 37.4 -> 31.4, P 19.9 -> 17.2, X' 61.6 -> 49.9
//   20 small matrices, a Muon step 759 -> 669
//
// Operands travel global -> LDS directly into swizzled 128-byte rows, as in
// the 256 x 256 kernel.  Rows past the matrix are read from its last row and
// the last k-tile's chunks past K from the row's last chunk; what they
// multiply is never stored, respectively zeroed in the fragments.
// kWide: rows so long that a tile's offsets need 64 bits.
template <typename Cfg, int kBlocksPerUnit, bool kWide>
__global__ __launch_bounds__(Cfg::kThreads, kBlocksPerUnit * Cfg::kWaves / 4) void gemm_nt_tiles_kernel(const TileLaunch launch) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  constexpr int TM = Cfg::TM, TN = Cfg::TN, KS = Cfg::KS, kDepth = Cfg::kDepth, kMfmas = TM * TN;
  constexpr int kLoadsA = Cfg::kLoadsA, kLoadsB = Cfg::kLoadsB;
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
  // An XCD with 64 tiles or more takes them in patches of eight rows, not four: over 8 x 8 tiles 16 operand panels
  // serve what takes 20 over 4 x 16.  Us with eight / four: 64 x 64 tiles 1424 x 1424, k 1424 18.5 / 19.6, 2000 x 2000
  // symmetric 25.1 / 26.5, 3064 x 824, k 824 14.2 / 13.8; 128 x 128 tiles 8 x 768 x 768 with 8 x 768 x 3072, k 768 49.9 /
  // 52.4, 3 x 4920 x 1032 54.7 / 53.3; 256 x 128 tiles 8 x 2080 x 2080 symmetric 88.3 / 89.5, 8 x 7696 x 1496 369 / 364.
  // Eight rows of the few tiles of a small launch cost it (14.7 -> 19.3).
  const int rows_together = p.items_per_xcd >= 64 ? 2 * kGroupTilesM : kGroupTilesM;
  if (!tile_of_workgroup(p, static_cast<int64_t>(blockIdx.x) - launch.first_workgroup[which], &batch, &tm, &tn, rows_together))
    return;  // whole workgroup
  batch = uniform_i64(batch);
  tm = uniform_i32(tm);
  tn = uniform_i32(tn);
  const int64_t m0 = static_cast<int64_t>(tm) * Cfg::BM, n0 = static_cast<int64_t>(tn) * Cfg::BN;

  // Load side: wave-level request q of an operand fills tile rows
  // [kFillRows q + 8 wave, +8); lane l fills slot l & 7 of row l >> 3 there.
  typedef std::conditional_t<kWide, uint64_t, uint32_t> offset_t;
  const int fill_row = 8 * wave + (lane >> 3);
  const int fill_chunk = (lane & 7) ^ ((fill_row >> 1) & 7);
  const uint8_t* a_src = uniform_ptr(reinterpret_cast<const uint8_t*>(p.A + batch * p.sA + m0 * p.lda));
  const uint8_t* b_src = uniform_ptr(reinterpret_cast<const uint8_t*>(p.B + batch * p.sB + n0 * p.ldb));
  offset_t a_voff[kLoadsA], b_voff[kLoadsB];
  const int a_last = static_cast<int>(p.M - m0 < Cfg::BM ? p.M - m0 : Cfg::BM) - 1;
  const int b_last = static_cast<int>(p.N - n0 < Cfg::BN ? p.N - n0 : Cfg::BN) - 1;
#pragma unroll
  for (int q = 0; q < kLoadsA; ++q)
    a_voff[q] = static_cast<offset_t>(min(Cfg::kFillRows * q + fill_row, a_last)) * static_cast<offset_t>(p.lda * 2) + fill_chunk * 16;
#pragma unroll
  for (int q = 0; q < kLoadsB; ++q)
    b_voff[q] = static_cast<offset_t>(min(Cfg::kFillRows * q + fill_row, b_last)) * static_cast<offset_t>(p.ldb * 2) + fill_chunk * 16;
  typedef __attribute__((address_space(3))) uint8_t* lds_address;
  const uint32_t fill_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_address)lds_bytes)) + wave * 1024;
  const int ktiles = static_cast<int>((p.K + Cfg::BK - 1) / Cfg::BK);
  const int tail = static_cast<int>(p.K / 8) & 7;  // chunks of the last k-tile, 0 if it is whole
  // Before the requests of the last k-tile: chunks past K read the row's last chunk instead.
  auto aim_at_tail = [&]() {
    const uint32_t back = fill_chunk >= tail ? (fill_chunk - (tail - 1)) * 16 : 0;
#pragma unroll
    for (int q = 0; q < kLoadsA; ++q) a_voff[q] -= back;
#pragma unroll
    for (int q = 0; q < kLoadsB; ++q) b_voff[q] -= back;
  };
  auto issue = [&](const uint8_t* src, offset_t voff, uint32_t slot, int q) {
    if constexpr (kWide) dma_load_16_at(src + voff, fill_lds + slot + q * (Cfg::kFillRows * Cfg::kRowBytes));
    else dma_load_16(voff, src, fill_lds + slot, q * (Cfg::kFillRows * Cfg::kRowBytes));
  };

  // Fragment side: lane l reads row l & 15 of a 16-row block, chunk 4 ks + (l >> 4).
  const int frag_row = lane & 15;
  const uint32_t frag_base = static_cast<uint32_t>(frag_row * Cfg::kRowBytes + (((lane >> 4) ^ ((frag_row >> 1) & 7)) * 16));
  uint32_t a_frag[KS], b_frag[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    a_frag[ks] = (frag_base ^ (ks * 64)) + wm * Cfg::kWaveM * Cfg::kRowBytes;
    b_frag[ks] = (frag_base ^ (ks * 64)) + wn * Cfg::kWaveN * Cfg::kRowBytes + Cfg::kARing;
  }
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 af[KS][TM], bf[KS][TN];
  // Fragment g of k step ks: the TM of operand A, then the TN of B.
  auto read_frag = [&](uint32_t a_slot, uint32_t b_slot, int ks, int g) {
    if (g < TM) af[ks][g] = *reinterpret_cast<const bf16x8*>(lds_bytes + a_slot + a_frag[ks] + g * 16 * Cfg::kRowBytes);
    else bf[ks][g - TM] = *reinterpret_cast<const bf16x8*>(lds_bytes + b_slot + b_frag[ks] + (g - TM) * 16 * Cfg::kRowBytes);
  };
  // Past K both operands are zero (the other's last values could be infinite).
  auto zero_past_k = [&](int ks) {
    const bool live = 4 * ks + (lane >> 4) < tail;
    const auto masked = [&](bf16x8& f) {
      const u32x4 w = __builtin_bit_cast(u32x4, f);
      f = __builtin_bit_cast(bf16x8, live ? w : u32x4{0, 0, 0, 0});
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) masked(af[ks][i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) masked(bf[ks][j]);
  };

  // One k-tile.  The barrier that hands over k-tile kt + 1 sits before the last
  // k step: that step's MFMAs cover the first fragment reads of kt + 1, and the
  // slot of B(kt) is free there (every wave holds its last fragments in registers).
  //   k step 0:     A(kt + kDepth) into the slot of A(kt - 1)
  //   wait for k-tile kt + 1, barrier
  //   k step 1:     B(kt + kDepth) into the slot of B(kt); kLateA: A(kt + kDepth), too, into the slot of A(kt)
  // Each step reads the next one's fragments.  A request goes out behind every
  // few MFMAs: several in one go hold up the wave.
  static_assert(KS == 2, "the sequence above");
  uint32_t a_slot = 0, b_slot = 0;  // of kt
  const auto next_of = [](uint32_t slot, uint32_t bytes, uint32_t ring) { return slot + bytes == ring ? 0u : slot + bytes; };
  constexpr int kReads = TM + TN, kReadSpan = kMfmas >= 2 * kReads ? kMfmas / 2 : kMfmas;
  // more: k-tile kt + 1 exists; ahead: kt + kDepth does.  a_src and b_src point at the latter.
  auto k_tile = [&](int kt, auto more_tag, auto ahead_tag) {
    constexpr bool more = decltype(more_tag)::value, ahead = decltype(ahead_tag)::value;
    const uint32_t a_next = next_of(a_slot, Cfg::kABytes, Cfg::kARing), b_next = next_of(b_slot, Cfg::kBBytes, Cfg::kBRing);
    const uint32_t a_before = a_slot == 0 ? Cfg::kARing - Cfg::kABytes : a_slot - Cfg::kABytes;
    // MFMA g of k step ks with what goes out behind it.
    auto slice = [&](int ks, int g) {
      const int i = g / TN, j = g % TN;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
      if (ks == 0 || more) {
#pragma unroll
        for (int r = 0; r < kReads; ++r)
          if (r * kReadSpan / kReads == g) {
            if (ks == 0) read_frag(a_slot, b_slot, 1, r);
            else read_frag(a_next, b_next, 0, r);
          }
      }
      if (ahead) {
        constexpr bool late = Cfg::kLateA;
        const int first = ks == 0 || late ? 0 : kLoadsA, last = ks == 0 ? (late ? 0 : kLoadsA) : Cfg::kLoads;
#pragma unroll
        for (int r = first; r < last; ++r)
          if ((r - first) * kMfmas / (last - first) == g) {
            if (r < kLoadsA) issue(a_src, a_voff[r], late ? a_slot : a_before, r);
            else issue(b_src, b_voff[r - kLoadsA], Cfg::kARing + b_slot, r - kLoadsA);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if (!more && tail) zero_past_k(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) slice(0, g);
    if (more) {
      // k-tile kt + 1 has landed (this wave's part); those behind it stay in flight.
      if (ahead) {
        wait_for_dma_loads_but<(kDepth - 2) * Cfg::kLoads + (Cfg::kLateA ? 0 : kLoadsA)>();
      } else {
        const int behind = ktiles - 2 - kt;
        if (kDepth >= 4 && behind == 2) wait_for_dma_loads_but<2 * Cfg::kLoads>();
        else if (kDepth >= 3 && behind == 1) wait_for_dma_loads_but<Cfg::kLoads>();
        else wait_for_dma_loads();
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else if (tail) {
      zero_past_k(1);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) slice(1, g);
    a_slot = a_next;
    b_slot = b_next;
    if (ahead) {
      a_src += Cfg::kRowBytes;
      b_src += Cfg::kRowBytes;
    }
  };

  // Fill the pipeline: the first kDepth k-tiles.
#pragma unroll
  for (int kt = 0; kt < kDepth; ++kt)
    if (kt < ktiles) {
      if (tail != 0 && kt == ktiles - 1) aim_at_tail();
#pragma unroll
      for (int q = 0; q < kLoadsA; ++q) issue(a_src, a_voff[q], kt * Cfg::kABytes, q);
#pragma unroll
      for (int q = 0; q < kLoadsB; ++q) issue(b_src, b_voff[q], Cfg::kARing + kt * Cfg::kBBytes, q);
      a_src += Cfg::kRowBytes;
      b_src += Cfg::kRowBytes;
    }
  if (kDepth >= 4 && ktiles >= 4) wait_for_dma_loads_but<3 * Cfg::kLoads>();
  else if (kDepth >= 3 && ktiles >= 3) wait_for_dma_loads_but<2 * Cfg::kLoads>();
  else if (ktiles >= 2) wait_for_dma_loads_but<Cfg::kLoads>();
  else wait_for_dma_loads();
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int g = 0; g < kReads; ++g) read_frag(0, 0, 0, g);
  __builtin_amdgcn_sched_barrier(0);
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  int kt = 0;
  for (; kt + kDepth < ktiles; ++kt) {
    if (tail != 0 && kt + kDepth == ktiles - 1) aim_at_tail();
    k_tile(kt, yes, yes);
  }
  for (; kt + 1 < ktiles; ++kt) k_tile(kt, yes, no);
  k_tile(ktiles - 1, no, no);
  __syncthreads();  // the images overlay the stages
  store_wave_tile<Cfg>(p, batch, m0 + wm * Cfg::kWaveM, n0 + wn * Cfg::kWaveN, lane, p.symmetric && tn >= p.symmetric * (tm + 1), acc,
                       lds_bytes + wave * Cfg::kRegion);
}

}  // namespace
}  // namespace fsh
