// Newton-Schulz orthogonalization for Muon on gfx950 matrix cores.
//
// Everything is built from one batched "NT" GEMM, C = bf16(alpha*A*B^T +
// beta*D) with both operands k-contiguous, so every MFMA operand is one
// 16-byte LDS read.  To keep all three products of an iteration in that
// form the iterate is carried in both orientations, X [s, l] and X^T [l, s]
// (s <= l):
//   G  = X X^T                 A = X,  B = X
//   P  = b G + c G G           A = G,  B = G   (G symmetric, so G^T = G)
//   X' = a X + P X             A = P,  B = X^T; the epilogue writes X' in
//                              place and X'^T into the other X^T buffer.
// A tall input is its own X^T, so no transpose kernel is needed in either
// case, and the result lands in the caller's buffer without a copy.
//
// GEMM kernels, operands global -> LDS directly: 256x256x64 tiles of 2x2
// wavefronts on v_mfma_f32_16x16x32_bf16 for large problems (below; those of
// Newton-Schulz need not be whole tiles), smaller tiles for everything else
// (gemm_tiles.hpp).
#include "gemm_tiles.hpp"
#include "muon_groups.hpp"


namespace fsh {
namespace {

// ---------------------------------------------------------------------------
// Large problems: 256x256x64 tiles with global->LDS loads.
//
// gfx950 can load 16 bytes per lane from global memory straight into LDS
// (global_load_lds_dwordx4: lane l of a wave writes LDS bytes
// [M0 + 16 l, M0 + 16 l + 16)), so a k-tile needs no staging registers and
// no ds_write.  A wave-level load fills 1 KB of LDS = 8 tile rows of 128 bytes
// with no padding, so bank conflicts are avoided by an XOR swizzle instead:
// the 16-byte chunk c of row r is stored in slot c ^ ((r >> 1) & 7) of its
// row, done on the global side by letting the lane that fills slot s of row r
// fetch chunk s ^ ((r >> 1) & 7).  The LDS has 64 banks of 4 bytes and serves
// a 16-byte-per-lane read sixteen lanes at a time; rows are 128 bytes, so the
// sixteen rows of such a group alternate between the two halves of the bank
// window and, within a half, take eight different slots.  (XOR with r & 7
// spreads only eight lanes and costs a two-way conflict on every fragment
// read: 8 instead of 4 cycles by the bank-conflict counter.)
//
// These loads and their waits are inline asm, which the compiler neither
// reorders nor counts; everything else in the loop is compiler-visible and is
// pinned around them with sched_barrier.
//
// The part does not hold its peak clock under this kernel: 1.84 GHz on random
// operands with the matrix cores 83 % busy (8192^3, by the counters).
struct DmaGemm {
  static constexpr int BM = 256, BN = 256, BK = 64, WM = 2, WN = 2;
  static constexpr int kThreads = 256, kWaveM = 128, kWaveN = 128;
  static constexpr int TM = kWaveM / 16, TN = kWaveN / 16, KS = BK / 32;  // 16x16x32 products
  static constexpr int kRowBytes = BK * 2;                   // 128
  static constexpr int kOperandBytes = BM * kRowBytes;       // 32 KB per operand and k-tile
  static constexpr int kSlots = 5;                           // ring of operand slots
  static constexpr int kRingBytes = kSlots * kOperandBytes;  // 160 KB, all of a compute unit's LDS
  static constexpr int kLoads = BM / 8 / 4;                  // wave-level 1 KB requests per wave and operand: 8
};

// LDS of the kernel: the ring; the epilogue's staging region lies from slot 2 upward.
constexpr int kDmaGemmLdsBytes = DmaGemm::kRingBytes;
constexpr int kDmaGemmStaging = 2 * DmaGemm::kOperandBytes;
static_assert(kDmaGemmStaging + HalfTileEpilogue<DmaGemm>::kLdsBytes <= kDmaGemmLdsBytes, "the epilogue works beside slots 0 and 1");

// (The empty statement keeps the cleared registers in place.)
__device__ __forceinline__ void clear_accumulators(f32x4& acc) {
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("" : "+a"(acc));
}

// kPersistent: the grid is one workgroup per compute unit and workgroup g
// takes the ids g, g + gridDim.x, ... of the launch (the same XCD every time,
// and the 32 workgroups of an XCD stay on 32 neighbouring tiles).  While the
// epilogue of a tile runs, the first operands of the next one are already on
// their way.  The schedule is static, so the host uses it only
// when all tiles of the launch are equally long; otherwise each id is its own
// workgroup and the hardware hands them out as compute units come free.
//
// kKMajor: both operands are given k-major, A as [K, M] and B as [K, N] (row
// strides lda / ldb), i.e. the product is A^T B.  A k-tile of an operand is
// then 64 rows of 512 bytes.  They land in LDS whole (the row order and the
// swizzle are at the load side below), and the fragments come out of it
// through the transposing LDS read of gfx950 (ds_read_b64_tr_b16): within 16
// lanes, lane 4 j + q passes the address of four consecutive columns 4 q ..
// 4 q + 3 of k-row j, and lane t receives column t of k-rows 0 .. 3 -- four
// consecutive k of one output row, half of an MFMA operand.  The products and
// their order are those of the k-contiguous form on the transposed operands,
// so the results are bit-identical.
//
// kRagged: some problem of the launch does not consist of whole tiles.  A
// separate instantiation: the limits in the epilogue and at a tile's start cost
// launches of whole tiles 1-2 %.
template <bool kPersistent, bool kKMajor, bool kRagged>
__global__ __launch_bounds__(DmaGemm::kThreads) void gemm_nt_dma_kernel(const GemmLaunch launch) {
  using Cfg = DmaGemm;
#ifdef FSH_TRACE
  const GemmParams& p = launch.problem[0];  // the profiling build stamps into the first problem's buffer
#endif
  FSH_STAMP(0);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_bytes[];
  constexpr int TM = Cfg::TM, TN = Cfg::TN, KS = Cfg::KS;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;

  // Tile of launch id `id`: problem index, batch, tile row and column (all
  // uniform; moved to scalar registers explicitly).  False for padding ids.
  auto locate = [&](int64_t id, int& which, int64_t& batch, int& tm, int& tn) -> bool {
    int w = 0;
#pragma unroll
    for (int i = 1; i < GemmLaunch::kMaxProblems; ++i) w += id >= launch.first_workgroup[i] ? 1 : 0;
    w = uniform_i32(w);
    int64_t b;
    int r, c;
    if (!tile_of_workgroup(launch.problem[w], id - launch.first_workgroup[w], &b, &r, &c)) return false;
    which = w;
    batch = uniform_i64(b);
    tm = uniform_i32(r);
    tn = uniform_i32(c);
    return true;
  };

  // Load side.  Wave-level load q (0..7) of this wave fills tile rows
  // [32 q + 8 wave, +8); lane l fills slot l & 7 of row l >> 3 there.
  // (k-major: load q fills k-rows r and r + 8, r = 16 (q / 2) + 4 (q % 2) + wave;
  // lane l fills slot l & 31 of row r + 8 (l >> 5).  K-row 16 a + 8 b + c thus
  // lies at byte 1024 (8 a + c) + 512 b of its slot.)
  // (The per-lane values of both sides are derived from the lane number again
  // at the start of every tile, see below.)
  uint32_t a_row_bytes = 0, b_row_bytes = 0;
  int a_left = 0, b_left = 0;  // rows of the operands from the tile's first on, 256 at most
  uint32_t a_voff[Cfg::kLoads], b_voff[Cfg::kLoads];
  const auto request_row = [](int q) -> int { return kKMajor ? 16 * (q / 2) + 4 * (q % 2) : 32 * q; };
  // M0 takes the LDS byte address relative to the workgroup's allocation.
  typedef __attribute__((address_space(3))) uint8_t* lds_address;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_address)lds_bytes));
  const uint32_t fill_lds = lds_base + static_cast<uint32_t>(wave * 1024);  // + q * 4096 + the ring slot
  // Operand tile bases of (problem, batch, tile row / column), k-tile 0.
  auto a_base = [&](int which, int64_t batch, int tm) -> const uint8_t* {
    const GemmParams& q = launch.problem[which];
    return uniform_ptr(reinterpret_cast<const uint8_t*>(
        q.A + batch * q.sA + static_cast<int64_t>(tm) * Cfg::BM * (kKMajor ? 1 : q.lda)));
  };
  auto b_base = [&](int which, int64_t batch, int tn) -> const uint8_t* {
    const GemmParams& q = launch.problem[which];
    return uniform_ptr(reinterpret_cast<const uint8_t*>(
        q.B + batch * q.sB + static_cast<int64_t>(tn) * Cfg::BN * (kKMajor ? 1 : q.ldb)));
  };
  // Request q of an operand's k-tile at `src` into the ring slot at `slot`.
  auto issue_one = [&](const uint8_t* src, const uint32_t (&voff)[Cfg::kLoads], int slot, int q) {
    dma_load_16(voff[q], src, slot + fill_lds, q * 4096);
  };
  auto issue_operand = [&](const uint8_t* src, const uint32_t (&voff)[Cfg::kLoads], int slot) {
#pragma unroll
    for (int q = 0; q < Cfg::kLoads; ++q) issue_one(src, voff, slot, q);
  };

  // Operand pointer of k-tile kt: 128 bytes along the rows, or 64 rows down.
  auto k_tile_ptr = [&](const uint8_t* base, uint32_t row_bytes, int64_t kt) -> const uint8_t* {
    return kKMajor ? base + kt * (static_cast<int64_t>(Cfg::BK) * row_bytes) : base + kt * Cfg::kRowBytes;
  };

  // Fragment side.  Lane l reads row l & 15 of a 16-row block, k chunk
  // 4 ks + (l >> 4); its slot is that chunk XOR ((row >> 1) & 7), i.e. the
  // ks = 0 address with bit 6 flipped by ks.
  uint32_t a_frag[KS], b_frag[KS];
  // k-major fragments: lane l = 16 g + t of a wave serves output row t of a
  // 16-row block and the k octet g of a k step; it passes the address of
  // columns 4 (t & 3) .. + 3 of k-row (t >> 2) of its octet's first half, then
  // of its second half (4 rows = 4096 bytes on).  The block index enters the
  // slot through the swizzle: chunk ^ 4 (k-row & 3) ^ 2 (octet & 1), one address
  // per block in the upper bits (i ^ (k-row & 3)) and two in the lower one.
  uint32_t a_frag_km[TM / 2][2], b_frag_km[TN / 2][2];
  // All per-lane addresses of the k loop are derived from the lane's number at
  // the start of every tile: the values then live from there to the end of the
  // k loop only.  Kept across the epilogue (which needs every register it can
  // get), the compiler spilled some of them and reloaded them inside the k
  // loop, and a reload is a vector memory load: the wait for it also waited
  // for every operand request in flight.
  // (So is that number itself, in two instructions.)
  const auto lane_now = []() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };
  // `octets` of a k-tile's eight exist.  What lies past the matrix is read from
  // its last row (k-major: column octet), what lies past K from the last octet:
  // the one is never stored, the other is zeroed in the fragments.
  auto derive_requests = [&](int l, int octets) {
    const int fill_row = kKMajor ? wave + 8 * (l >> 5) : 8 * wave + (l >> 3);
    // (k-row & 3 of a k-major request is the wave's number)
    const int fill_chunk = kKMajor ? (l & 31) ^ (4 * wave) ^ (2 * (l >> 5)) : (l & 7) ^ ((fill_row >> 1) & 7);
    const auto offset = [&](int q, int left, uint32_t row_bytes) {
      const int row = fill_row + request_row(q);
      const int row_there = !kRagged ? row : kKMajor ? min(row, 8 * octets - 1) : min(row, left - 1);
      const int chunk_there = !kRagged ? fill_chunk : kKMajor ? min(fill_chunk, left / 8 - 1) : min(fill_chunk, octets - 1);
      return static_cast<uint32_t>(row_there) * row_bytes + static_cast<uint32_t>(chunk_there * 16);
    };
#pragma unroll
    for (int q = 0; q < Cfg::kLoads; ++q) {
      a_voff[q] = offset(q, a_left, a_row_bytes);
      b_voff[q] = offset(q, b_left, b_row_bytes);
    }
  };
  auto derive_fragments = [&](int l) {
    const int t = l & 15, g = l >> 4;
    const uint32_t frag_base = static_cast<uint32_t>(t * Cfg::kRowBytes + ((g ^ ((t >> 1) & 7)) * 16));
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      a_frag[ks] = (frag_base ^ (ks * 64)) + wm * Cfg::kWaveM * Cfg::kRowBytes;
      b_frag[ks] = (frag_base ^ (ks * 64)) + wn * Cfg::kWaveN * Cfg::kRowBytes;
    }
    const uint32_t common = static_cast<uint32_t>((g >> 1) * 8192 + (t >> 2) * 1024 + (g & 1) * 512 + (t & 3) * 8);
#pragma unroll
    for (int i = 0; i < TM / 2; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) a_frag_km[i][e] = common + wm * 256 + ((i ^ (t >> 2)) * 64) + ((e ^ (g & 1)) * 32);
#pragma unroll
    for (int j = 0; j < TN / 2; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) b_frag_km[j][e] = common + wn * 256 + ((j ^ (t >> 2)) * 64) + ((e ^ (g & 1)) * 32);
  };
  f32x4 acc[TM][TN];
  bf16x8 af[2][TM], bf[2][TN];
  auto read_transposed = [&](uint32_t offset) -> bf16x8 {
    typedef short i16x4 __attribute__((__vector_size__(4 * sizeof(short))));
    typedef __attribute__((address_space(3))) i16x4* lds_i16x4;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)(lds_bytes + offset));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)(lds_bytes + offset + 4096));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto read_a = [&](int set, int slot, int ks, int i) {
    if (kKMajor)
      af[set][i] = read_transposed(slot + a_frag_km[i / 2][i % 2] + ks * 16384);
    else
      af[set][i] = *reinterpret_cast<const bf16x8*>(lds_bytes + slot + a_frag[ks] + i * 16 * Cfg::kRowBytes);
  };
  auto read_b = [&](int set, int slot, int ks, int j) {
    if (kKMajor)
      bf[set][j] = read_transposed(slot + b_frag_km[j / 2][j % 2] + ks * 16384);
    else
      bf[set][j] = *reinterpret_cast<const bf16x8*>(lds_bytes + slot + b_frag[ks] + j * 16 * Cfg::kRowBytes);
  };
  // Fragment g of k step ks: the TM of operand A, then the TN of B.
  auto read_frag = [&](int set, int a_slot, int b_slot, int ks, int g) {
    if (g < TM) read_a(set, a_slot, ks, g);
    else read_b(set, b_slot, ks, g - TM);
  };
  auto mfma = [&](int set, int i, int j) {
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[set][j], af[set][i], acc[i][j], 0, 0, 0);
  };
  // Current tile: plain scalars, reassigned per tile.
  int which = 0, tm = 0, tn = 0;
  int64_t batch = 0;
  int64_t id = blockIdx.x;
  const int64_t stride = gridDim.x;
  if (kPersistent) {
    while (id < launch.total_workgroups && !locate(id, which, batch, tm, tn)) id = uniform_i64(id + stride);
    if (id >= launch.total_workgroups) return;  // whole workgroup, before any barrier
  } else if (!locate(id, which, batch, tm, tn)) {
    return;  // whole workgroup, before any barrier
  }
  const uint8_t* Ab = nullptr;
  const uint8_t* Bb = nullptr;
  // The first operands of a tile, into slots 0 and 1.
  auto begin_tile = [&](int problem, int64_t matrix, int r, int c) {
    const GemmParams& q = launch.problem[problem];
    Ab = a_base(problem, matrix, r);
    Bb = b_base(problem, matrix, c);
    a_row_bytes = static_cast<uint32_t>(q.lda * 2);
    b_row_bytes = static_cast<uint32_t>(q.ldb * 2);
    if (kRagged) {
      const int64_t m_left = q.M - static_cast<int64_t>(r) * Cfg::BM, n_left = q.N - static_cast<int64_t>(c) * Cfg::BN;
      a_left = static_cast<int>(m_left < Cfg::BM ? m_left : Cfg::BM);
      b_left = static_cast<int>(n_left < Cfg::BN ? n_left : Cfg::BN);
    }
    derive_requests(lane_now(), 8);  // (a contraction that ends inside a k-tile has at least three)
    issue_operand(Ab, a_voff, 0);
    issue_operand(Bb, b_voff, Cfg::kOperandBytes);
  };
  FSH_STAMP(1);
  begin_tile(which, batch, tm, tn);

#ifdef FSH_TRACE
  uint64_t trace_wait = 0, trace_barrier = 0, trace_ktiles = 0, trace_tile_wait = 0, trace_tile_barrier = 0, trace_tiles = 0, trace_kloop = 0, trace_epi = 0, trace_steps = 0, trace_last = 0, trace_mark = 0;
  const uint64_t trace_begin = __builtin_amdgcn_s_memtime();
#endif
  // The k loop.  What bounds it: power, then the issue slots of the one wave
  // per SIMD.  The request path of a compute unit takes one of the 64 requests
  // of a k-tile (16 per wave) per 16 cycles, so they need half of the 2048
  // cycles of the MFMAs, and a wave that issues a request into a busy path
  // cannot issue MFMAs.  Packed into half of the k-tile, as two 64 KB stages
  // ask for (a stage is free only once the k-tile in it has been read), they
  // cost 500 of the 3000 cycles a k-tile took, and the wait for the last ones
  // up to 460.  The ring holds two and a half k-tiles instead: operand n of the
  // sequence A(0), B(0), A(1), B(1), ... lives in slot n % 5, so A is requested
  // two k-tiles ahead while both operands of the next one are still on their
  // way, and a request goes out every eighth MFMA.
  //
  // The barrier that hands over k-tile kt + 1 sits before the last k step of
  // kt: that step's MFMAs cover the first fragment reads of kt + 1, and the
  // slots of kt are free (every wave holds its last fragments in registers).
  //   k step 0:     A(kt + 2) into the fifth slot
  //   wait for all but A(kt + 2), barrier
  //   k step 1:     B(kt + 2) into the slot of A(kt)
  // Each step reads the next one's fragments.
  //
  // 16x16x32 MFMAs read and write half as many accumulators per product as
  // 32x32x16 ones and draw less power for it: the part then runs this loop at
  // 1.84 instead of 1.67 GHz.
  // Us with two stages and 32x32x16 / ring / ring and 16x16x32:
  //   24 x 7168 x 2048, k 2048 1327 / 1190 / 1115    8192^3 901 / 821 / 755   4096^3 108 / 104 / 93
  //   24 x 2048 x 2048, k 7168, k-major and symmetric 786 / 728 / 712
  // Where in its step a request or a read goes out, and the order of the
  // MFMAs, matter by 1 %: two rows of blocks at a time is the best by that.
  constexpr int kMfmas = TM * TN, kReadEvery = 2;  // a fragment read behind every second MFMA
  static_assert(KS == 2, "the sequence above");
  const auto next_slot = [](int slot) { return slot + Cfg::kOperandBytes == Cfg::kRingBytes ? 0 : slot + Cfg::kOperandBytes; };
  int a_slot = 0;  // of the current k-tile's operand A
  // more: k-tile kt + 1 exists; more2: kt + 2 exists
  int tail = 0;  // octets of the last k-tile, 0 if it is whole
  auto k_tile = [&](int kt, auto more_tag, auto more2_tag) {
    constexpr bool more = decltype(more_tag)::value, more2 = decltype(more2_tag)::value;
    const int b_slot = next_slot(a_slot), a_next = next_slot(b_slot), b_next = next_slot(a_next), a_after = next_slot(b_next);
    const uint8_t* a_src2 = k_tile_ptr(Ab, a_row_bytes, kt + 2);
    const uint8_t* b_src2 = k_tile_ptr(Bb, b_row_bytes, kt + 2);
    // MFMA g of k step ks with what goes out behind it.
    auto slice = [&](int ks, int g) {
      mfma(ks, g / (2 * TN) * 2 + g % 2, g % (2 * TN) / 2);
      if (g % kReadEvery == kReadEvery - 1 && g / kReadEvery < TM + TN) {
        if (ks == 0) read_frag(1, a_slot, b_slot, 1, g / kReadEvery);
        else if (more) read_frag(0, a_next, b_next, 0, g / kReadEvery);
      }
      if ((g + 1) % (kMfmas / Cfg::kLoads) == 0 && more2) {
        const int r = g / (kMfmas / Cfg::kLoads);
        if (ks == 0) issue_one(a_src2, a_voff, a_after, r);
        else issue_one(b_src2, b_voff, a_slot, r);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // Past K both operands are zero (the other's last values could be infinite).
    auto zero_past_k = [&](int ks) {
      const bool live = 4 * ks + (lane_now() >> 4) < tail;
      const auto masked = [&](bf16x8& f) {
        const u32x4 w = __builtin_bit_cast(u32x4, f);
        f = __builtin_bit_cast(bf16x8, live ? w : u32x4{0, 0, 0, 0});
      };
#pragma unroll
      for (int i = 0; i < TM; ++i) masked(af[ks][i]);
#pragma unroll
      for (int j = 0; j < TN; ++j) masked(bf[ks][j]);
    };
    if (kRagged && !more && tail) zero_past_k(0);
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) slice(0, g);
    if (kRagged && !more && tail) zero_past_k(1);
#ifdef FSH_TRACE
    const uint64_t tr0 = __builtin_amdgcn_s_memtime();
    trace_steps += tr0 - trace_mark;
#endif
    // This wave's part of k-tile kt + 1 has landed; A(kt + 2) stays in flight.
    if (more2) wait_for_dma_loads_but<Cfg::kLoads>();
    else if (more) wait_for_dma_loads();
#ifdef FSH_TRACE
    const uint64_t tr1 = __builtin_amdgcn_s_memtime();
#endif
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#ifdef FSH_TRACE
    const uint64_t tr2 = __builtin_amdgcn_s_memtime();
    trace_wait += tr1 - tr0;
    trace_barrier += tr2 - tr1;
    trace_ktiles += 1;
#endif
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) slice(1, g);
    a_slot = a_next;
#ifdef FSH_TRACE
    trace_mark = __builtin_amdgcn_s_memtime();
    trace_last += trace_mark - tr2;
#endif
  };

  while (true) {
    const GemmParams& p = launch.problem[which];
    const int ktiles = static_cast<int>((p.K + Cfg::BK - 1) / Cfg::BK);
    if (kRagged) tail = static_cast<int>(p.K / 8) & 7;
    derive_requests(lane_now(), 8);
    derive_fragments(lane_now());
    FSH_STAMP(6);
    // Under the wait for the first operands and for the previous tile's stores.
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) clear_accumulators(acc[g / TN][g % TN]);
#ifdef FSH_TRACE
    const uint64_t ts0 = __builtin_amdgcn_s_memtime();
#endif
    wait_for_dma_loads();
    FSH_STAMP(7);
#ifdef FSH_TRACE
    const uint64_t ts1 = __builtin_amdgcn_s_memtime();
#endif
    __syncthreads();  // also: every wave has left the previous tile's epilogue
#ifdef FSH_TRACE
    trace_tile_wait += ts1 - ts0;
    trace_tile_barrier += __builtin_amdgcn_s_memtime() - ts1;
    trace_tiles += 1;
    const uint64_t tk0 = __builtin_amdgcn_s_memtime();
    trace_mark = tk0;
#endif
    a_slot = 0;
#pragma unroll
    for (int g = 0; g < TM + TN; ++g) read_frag(0, 0, Cfg::kOperandBytes, 0, g);
    if (ktiles > 1) {
      issue_operand(k_tile_ptr(Ab, a_row_bytes, 1), a_voff, 2 * Cfg::kOperandBytes);
      issue_operand(k_tile_ptr(Bb, b_row_bytes, 1), b_voff, 3 * Cfg::kOperandBytes);
    }
    FSH_STAMP(2);

    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    for (int kt = 0; kt + 2 < ktiles; ++kt) {
      if (kRagged && kt + 3 == ktiles && tail) derive_requests(lane_now(), tail);  // the last k-tile's go out in this one
      k_tile(kt, yes, yes);
    }
    if (ktiles > 1) k_tile(ktiles - 2, yes, no);
    k_tile(ktiles - 1, no, no);
    FSH_STAMP(3);
#ifdef FSH_TRACE
    trace_kloop += __builtin_amdgcn_s_memtime() - tk0;
#endif

    // All slots are free now.  The next tile's first operands go to slots 0 and
    // 1 while the epilogue stages its output beside them.
    int next_which = 0, next_tm = 0, next_tn = 0;
    int64_t next_batch = 0;
    bool have_next = false;
    if (kPersistent) {
      id = uniform_i64(id + stride);
      while (id < launch.total_workgroups && !(have_next = locate(id, next_which, next_batch, next_tm, next_tn)))
        id = uniform_i64(id + stride);
      if (have_next) begin_tile(next_which, next_batch, next_tm, next_tn);
    }
#ifdef FSH_TRACE
    const uint64_t te0 = __builtin_amdgcn_s_memtime();
#endif
    store_tile_in_halves<Cfg, kRagged>(p, batch, static_cast<int64_t>(tm) * Cfg::BM, static_cast<int64_t>(tn) * Cfg::BN, wm,
                              wn, lane_now(), p.symmetric && tm != tn, acc, lds_bytes + kDmaGemmStaging);
#ifdef FSH_TRACE
    trace_epi += __builtin_amdgcn_s_memtime() - te0;
#endif
    FSH_STAMP(4);
#if defined(FSH_TRACE) && !defined(FSH_TRACE_NODRAIN)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    FSH_STAMP(5);
#endif
#ifdef FSH_TRACE
    if (!have_next && p.trace && threadIdx.x == 0) {
      p.trace[blockIdx.x * 16 + 12] = __builtin_amdgcn_s_memtime() - trace_begin;
      p.trace[blockIdx.x * 16 + 13] = trace_wait;
      p.trace[blockIdx.x * 16 + 14] = trace_barrier;
      p.trace[blockIdx.x * 16 + 15] = trace_ktiles;
      p.trace[blockIdx.x * 16 + 8] = trace_tile_wait;
      p.trace[blockIdx.x * 16 + 9] = trace_tile_barrier;
      p.trace[blockIdx.x * 16 + 10] = trace_tiles;
      p.trace[blockIdx.x * 16 + 11] = trace_kloop;
      p.trace[blockIdx.x * 16 + 7] = trace_epi;
      p.trace[blockIdx.x * 16 + 5] = trace_steps;
      p.trace[blockIdx.x * 16 + 6] = trace_last;
    }
#endif
    if (!have_next) break;
    which = next_which;
    batch = next_batch;
    tm = next_tm;
    tn = next_tn;
  }
}

// A validated problem, whether the large-tile kernel can take it and whether it does.
struct PlannedGemm {
  GemmParams p;
  int64_t batch;
  bool fits, large;
};

// ---- Which tiles a launch takes.
// Measured at k = 512 / 2048 (us; k-tiles of 64; 128 x 128: where one workgroup
// per compute unit would do, the deep form in brackets):
//               64 x 64       128 x 128                   256 x 128      256 x 256
//   1024 x 1024    5.0 /  9.6    6.9 / 14.8 ( 7.5 / 15.3)    8.9 / 23.8   15.3 / 37.5
//   2048 x 2048    8.9 / 25.9    8.0 / 21.2 ( 8.5 / 18.4)    9.8 / 24.3   16.0 / 38.6
//   4096 x 2048   15.4 / 47.3   12.4 / 31.4                 12.2 / 29.9   17.7 / 39.8
//   4096 x 4096   28.4 / 90.0   21.7 / 58.7                 23.2 / 57.9   19.9 / 49.8
// The constants below were fitted to earlier kernels of the three smaller sizes
// (4096 x 4096, k 2048: 108.5, 80.5, 74.6).  Over 50 products of 256 to 8192 a
// side the estimates are now, as a multiple of the measured time (tenth, middle
// and ninth of ten), for rows at cache lines 1.06 / 1.23 / 1.36, 1.13 / 1.25 / 1.38,
// deep 0.96 / 1.07 / 1.19, 1.09 / 1.19 / 1.31 and 0.90 / 0.96 / 1.05, and lower by a
// tenth for rows that straddle them: beside the others the deep tiles and the
// 256 x 256 ones look better than they are.  None of 80 products and 50 Muon
// steps was slower for it than with the earlier kernels; the fastest kind would
// have been 3 % faster in the mean.
enum TileKind { kTiles64, kTiles128, kTiles128Deep, kTiles256x128, kTiles256 };  // the order of kTileShapes
constexpr int kTileNames[] = {FSH_TILES_64, FSH_TILES_128, FSH_TILES_128_DEEP, FSH_TILES_256X128, FSH_TILES_256};
constexpr TileShape kTileShapes[] = {
    {64, 64, 768.0, 0.17, 0.40, 0.55, 1.7},       // three workgroups per compute unit (four fit)
    {128, 128, 512.0, 0.37, 0.71, 1.02, 4.2},     // two
    {128, 128, 256.0, 0.35, 0.43, 0.52, 3.2},     // one, its operands requested four k-tiles ahead
    {256, 128, 256.0, 0.54, 0.68, 0.91, 5.5},     // one of eight waves
    {256, 256, 256.0, 0.94, 1.02, 1.38, 8.5},     // one
};
// The products of one launch, as the tiles of every kind see them.
struct LaunchWork {
  double tiles[5] = {0, 0, 0, 0, 0}, tile_ktiles[5] = {0, 0, 0, 0, 0};
  double max_ktiles = 0.0;
  bool transposed = false;  // some product is written transposed as well
  void add(int64_t m, int64_t n, int64_t k, bool symmetric, int64_t batch);
};
int64_t count_tiles(int64_t m, int64_t n, bool symmetric, int64_t tile_m, int64_t tile_n) {
  const int64_t tm = ceil_div(m, tile_m), tn = ceil_div(n, tile_n), step = tile_m / tile_n;
  return symmetric ? tm * tn - step * (tm * (tm - 1) / 2) : tm * tn;
}
void LaunchWork::add(int64_t m, int64_t n, int64_t k, bool symmetric, int64_t batch) {
  const double kt = static_cast<double>(ceil_div(k, (int64_t)64));
  for (int i = 0; i < 5; ++i) {
    const double count = static_cast<double>(count_tiles(m, n, symmetric, kTileShapes[i].m, kTileShapes[i].n)) * static_cast<double>(batch);
    tiles[i] += count;
    tile_ktiles[i] += count * kt;
  }
  max_ktiles = fmax(max_ktiles, kt);
}
// Tiles of a shorter contraction count by their share of the longest one.
double launch_us(TileKind kind, const LaunchWork& w) {
  if (w.max_ktiles == 0.0) return 0.0;
  // A second output lengthens the end of every round: 128 KB more of each 256 x 256 tile leave at a time.
  TileShape shape = kTileShapes[kind];
  if (w.transposed) shape.ends += kind == kTiles256 ? 12.0 : 3.0;
  return rounds_us(shape, w.tiles[kind], w.tile_ktiles[kind], w.max_ktiles);
}
TileKind small_tile_kind(const LaunchWork& w) {
  TileKind best = kTiles64;
  for (const TileKind kind : {kTiles128, kTiles128Deep, kTiles256x128}) {
    // One round or none; short tiles beside longer ones count by their length there, up to 0.86 of a round of them:
    // the hand-out is not that even.  Muon steps, us without / with such mixtures, by the part of a round: 0.81 (13 of
    // 3555 x 384, 2432 x 2432) 790 / 727, 0.84 (4 of 1024 x 4096, 8 of 1024 x 1024) 690 / 674, 0.87 (8 of 768 x 768, 4
    // each of 3072 x 768 and 768 x 3072, four odd ones) 617 / 620, 1.0 (2 of 1280 x 1280, 8 of 832 x 832) 380 / 406.
    if (kind == kTiles128Deep && w.tiles[kind] > kTileShapes[kind].round &&
        w.tile_ktiles[kind] > 0.86 * kTileShapes[kind].round * w.max_ktiles)
      continue;
    if (launch_us(kind, w) < launch_us(best, w)) best = kind;
  }
  return best;
}
constexpr double kEstimateMargin = 0.95;  // for the error of the comparison (see above: it favours the large tiles)
double small_tiles_us(const LaunchWork& w) { return launch_us(small_tile_kind(w), w); }

// The 256 x 256 kernel has 16-byte accesses in the epilogue and 32-bit tile spans.
// It aims its requests at a k-tile that the contraction ends in only inside the
// k loop, two k-tiles ahead: with the tile's third at the earliest.
bool fits_large_tiles(const GemmParams& p) {
  return p.M % 8 == 0 && p.N % 8 == 0 && p.K % 8 == 0 && (p.K % DmaGemm::BK == 0 || p.K > 2 * DmaGemm::BK) && p.ldc % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && p.sC % 8 == 0 &&
         (p.Ct == nullptr || (p.ldct % 8 == 0 && (reinterpret_cast<uintptr_t>(p.Ct) & 15) == 0 && p.sCt % 8 == 0)) &&
         (p.D == nullptr || (p.ldd % 8 == 0 && (reinterpret_cast<uintptr_t>(p.D) & 15) == 0 && p.sD % 8 == 0)) &&
         static_cast<int64_t>(DmaGemm::BM) * p.lda * 2 < (1LL << 31) && static_cast<int64_t>(DmaGemm::BN) * p.ldb * 2 < (1LL << 31);
}
bool whole_large_tiles(const GemmParams& p) {
  return p.M % DmaGemm::BM == 0 && p.N % DmaGemm::BN == 0 && p.K % DmaGemm::BK == 0;
}

// The Muon update an epilogue applies instead of storing its product (see
// GemmParams::update_ptrs); ptrs == nullptr: an ordinary product.
struct GemmUpdate {
  const int64_t* ptrs;
  float decay, neg_lr, dir_scale;
};

int plan_gemm(const fsh_gemm_desc& d, PlannedGemm* plan, const GemmUpdate* update = nullptr) {
  if (d.m <= 0 || d.n <= 0 || d.k <= 0 || d.batch <= 0)
    return fail(FSH_EINVAL, "gemm: non-positive size (m %lld, n %lld, k %lld, batch %lld)", (long long)d.m,
                (long long)d.n, (long long)d.k, (long long)d.batch);
  if (!d.a_dev || !d.b_dev || !d.c_dev) return fail(FSH_EINVAL, "gemm: null operand");
  if (d.k % 8 || d.lda % 8 || d.ldb % 8 || d.stride_a % 8 || d.stride_b % 8 || !aligned(d.a_dev, 16) ||
      !aligned(d.b_dev, 16))
    return fail(FSH_ENOTSUP, "gemm: k, lda, ldb and batch strides must be multiples of 8 and A, B 16-byte aligned");
  // k-contiguous operands have rows of k elements; k-major ones rows of m and of n.
  if (d.lda < (d.k_major ? d.m : d.k) || d.ldb < (d.k_major ? d.n : d.k) || d.ldc < d.n || (d.d_dev && d.ldd < d.n) ||
      (d.ct_dev && d.ldct < d.m))
    return fail(FSH_EINVAL, "gemm: leading dimension smaller than the row length");
  if (d.symmetric && (d.m != d.n || d.ct_dev != nullptr))
    return fail(FSH_EINVAL, "gemm: a symmetric product needs m == n and no transposed output");
  GemmParams& p = plan->p;
  memset(&p, 0, sizeof(p));
  p.symmetric = d.symmetric ? 1 : 0;
  p.k_major = d.k_major ? 1 : 0;
  p.A = static_cast<const uint16_t*>(d.a_dev);
  p.B = static_cast<const uint16_t*>(d.b_dev);
  p.D = static_cast<const uint16_t*>(d.d_dev);
  p.C = static_cast<uint16_t*>(d.c_dev);
  p.Ct = static_cast<uint16_t*>(d.ct_dev);
  p.M = d.m; p.N = d.n; p.K = d.k;
  p.lda = d.lda; p.ldb = d.ldb; p.ldd = d.ldd; p.ldc = d.ldc; p.ldct = d.ldct;
  p.sA = d.stride_a; p.sB = d.stride_b; p.sD = d.stride_d; p.sC = d.stride_c; p.sCt = d.stride_ct;
  p.alpha = d.alpha; p.beta = d.beta;
  p.diag_add = d.diag_add;
  if (update != nullptr && update->ptrs != nullptr) {
    if (d.d_dev != nullptr || d.ct_dev != nullptr || d.symmetric || d.alpha != 1.0f || d.diag_add != 0.0f)
      return fail(FSH_EINVAL, "gemm: a fused update takes a plain product");
    p.update_ptrs = update->ptrs;
    p.update_decay = update->decay;
    p.update_neg_lr = update->neg_lr;
    p.update_dir_scale = update->dir_scale;
  }
#ifdef FSH_TRACE
  if (const char* e = getenv("FSH_GEMM_TRACE")) p.trace = reinterpret_cast<uint64_t*>(strtoull(e, nullptr, 0));
#endif
  plan->batch = d.batch;
  plan->fits = fits_large_tiles(p);
  plan->large = plan->fits && whole_large_tiles(p);  // may take the large-tile kernel; choose_kernels decides whether it does
  return FSH_OK;
}


// Which of the problems that may take the large-tile kernel do: all of them
// (together they fill its launch) or none, whichever is estimated to take
// less time with the rest of the call.  Operands given k-major and fused
// updates exist in the large-tile kernel only.
int choose_kernels(PlannedGemm* plans, int count) {
  LaunchWork large, small, all;
  bool bound = false;
  for (int i = 0; i < count; ++i) {
    const GemmParams& p = plans[i].p;
    const bool must = p.k_major || p.update_ptrs != nullptr;
    if (must && !plans[i].large)
      return fail(FSH_ENOTSUP, "gemm: k-major operands and fused updates need whole 256 x 256 x 64 tiles (m %lld, n %lld, k %lld)",
                  (long long)p.M, (long long)p.N, (long long)p.K);
    bound = bound || must;
    all.add(p.M, p.N, p.K, p.symmetric != 0, plans[i].batch);
    (plans[i].large ? large : small).add(p.M, p.N, p.K, p.symmetric != 0, plans[i].batch);
  }
  if (!bound && small_tiles_us(all) <= launch_us(kTiles256, large) + small_tiles_us(small))
    for (int i = 0; i < count; ++i) plans[i].large = false;
  return FSH_OK;
}

// Fills in a problem's schedule of tile_m x tile_n tiles.
int schedule_tiles(PlannedGemm* plan, int64_t tile_m, int64_t tile_n, int64_t* workgroups) {
  GemmParams& p = plan->p;
  const int64_t tiles_m = ceil_div(p.M, tile_m), tiles_n = ceil_div(p.N, tile_n);
  const int64_t tiles = count_tiles(p.M, p.N, p.symmetric != 0, tile_m, tile_n);
  if (p.symmetric) p.symmetric = static_cast<int32_t>(tile_m / tile_n);
  p.work_items = tiles * plan->batch;
  p.items_per_xcd = ceil_div(p.work_items, static_cast<int64_t>(kXcds));
  if (tiles > 0x3FFFFFFFLL || p.items_per_xcd * kXcds > 0x3FFFFFFFLL) return fail(FSH_ENOTSUP, "gemm: too many tiles");
  p.tiles_m = static_cast<int32_t>(tiles_m);
  p.tiles_n = static_cast<int32_t>(tiles_n);
  p.tiles_per_matrix = static_cast<int32_t>(tiles);
  *workgroups = p.items_per_xcd * kXcds;
  return FSH_OK;
}

// The problems `members` (indices into plans, longest k first) as one launch of tile_m x tile_n tiles.
template <typename Launch>
int fill_launch(PlannedGemm* plans, const int* members, int n, int64_t tile_m, int64_t tile_n, Launch* launch) {
  memset(launch, 0, sizeof(*launch));
  int64_t first = 0;
  for (int k = 0; k < Launch::kMaxProblems; ++k) {
    launch->first_workgroup[k] = INT32_MAX;
    if (k >= n) continue;
    int64_t workgroups = 0;
    if (int rc = schedule_tiles(&plans[members[k]], tile_m, tile_n, &workgroups)) return rc;
    launch->first_workgroup[k] = static_cast<int32_t>(first);
    launch->problem[k] = plans[members[k]].p;
    first += workgroups;
    if (first > 0x3FFFFFFFLL) return fail(FSH_ENOTSUP, "gemm: too many tiles in one launch");
  }
  launch->total_workgroups = static_cast<int32_t>(first);
  return FSH_OK;
}

template <bool kPersistent, bool kKMajor, bool kRagged>
int launch_large_as(const GemmLaunch& launch, int64_t workgroups, hipStream_t stream) {
  static LdsReservation reserved;
  constexpr auto* kernel = &gemm_nt_dma_kernel<kPersistent, kKMajor, kRagged>;
  if (int rc = reserve_lds_once(reserved, kernel, kDmaGemmLdsBytes)) return rc;
  hipLaunchKernelGGL((gemm_nt_dma_kernel<kPersistent, kKMajor, kRagged>), dim3(static_cast<uint32_t>(workgroups)),
                     dim3(DmaGemm::kThreads), kDmaGemmLdsBytes, stream, launch);
  return check_launch("gemm_nt_dma_kernel");
}
int launch_large_tiles(const GemmLaunch& launch, bool k_major, hipStream_t stream) {
  // Equally long tiles and more of them than compute units: one resident
  // workgroup per compute unit walks a static schedule.
  bool equal_k = true, ragged = false;
  for (int k = 0; k < GemmLaunch::kMaxProblems; ++k) {
    if (launch.first_workgroup[k] == INT32_MAX) continue;
    equal_k = equal_k && launch.problem[k].K == launch.problem[0].K;
    ragged = ragged || !whole_large_tiles(launch.problem[k]);
  }
  const int64_t units = compute_units(), total = launch.total_workgroups;
  const bool resident = equal_k && units >= kXcds && units % kXcds == 0 && total > units;
  const int64_t workgroups = resident ? units : total;
  switch ((resident ? 4 : 0) + (k_major ? 2 : 0) + (ragged ? 1 : 0)) {
    case 0: return launch_large_as<false, false, false>(launch, workgroups, stream);
    case 1: return launch_large_as<false, false, true>(launch, workgroups, stream);
    case 2: return launch_large_as<false, true, false>(launch, workgroups, stream);
    case 3: return launch_large_as<false, true, true>(launch, workgroups, stream);
    case 4: return launch_large_as<true, false, false>(launch, workgroups, stream);
    case 5: return launch_large_as<true, false, true>(launch, workgroups, stream);
    case 6: return launch_large_as<true, true, false>(launch, workgroups, stream);
    default: return launch_large_as<true, true, true>(launch, workgroups, stream);
  }
}

template <typename Cfg, int kBlocksPerUnit, bool kWide = false>
int launch_tiles_as(const TileLaunch& launch, hipStream_t stream) {
  static LdsReservation reserved;
  constexpr auto* kernel = &gemm_nt_tiles_kernel<Cfg, kBlocksPerUnit, kWide>;
  if (int rc = reserve_lds_once(reserved, kernel, Cfg::kLdsBytes)) return rc;
  hipLaunchKernelGGL((gemm_nt_tiles_kernel<Cfg, kBlocksPerUnit, kWide>), dim3(static_cast<uint32_t>(launch.total_workgroups)),
                     dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, launch);
  return check_launch("gemm_nt_tiles_kernel");
}

LaunchWork work_of(const PlannedGemm* plans, const int* members, int n) {
  LaunchWork work;
  for (int k = 0; k < n; ++k) {
    const GemmParams& p = plans[members[k]].p;
    work.add(p.M, p.N, p.K, p.symmetric != 0, plans[members[k]].batch);
  }
  return work;
}

// Rows so long that the operand offsets of a tile of any kind need 64 bits.
bool has_wide_rows(const PlannedGemm* plans, const int* members, int n) {
  for (int k = 0; k < n; ++k) {
    const GemmParams& p = plans[members[k]].p;
    if (256 * 2 * (p.lda > p.ldb ? p.lda : p.ldb) >= (1LL << 31)) return true;
  }
  return false;
}
// Whether three quarters of a launch's work on tiles of a kind read operand rows
// that do not start at cache lines: a k-tile's 128 bytes of such a row touch two.
// (With six tenths, 5 of 952 x 1128 beside whole rows, a Muon step takes 438 us as
// the others and 443 as these; with a half 584 and 587.)
bool has_split_rows(const PlannedGemm* plans, const int* members, int n, TileKind kind) {
  double split = 0.0, all = 0.0;
  for (int k = 0; k < n; ++k) {
    const GemmParams& p = plans[members[k]].p;
    LaunchWork work;
    work.add(p.M, p.N, p.K, p.symmetric != 0, plans[members[k]].batch);
    all += work.tile_ktiles[kind];
    const auto at_lines = [&](const uint16_t* rows, int64_t ld, int64_t stride) {
      return aligned(rows, 128) && ld % 64 == 0 && (plans[members[k]].batch == 1 || stride % 64 == 0);
    };
    if (!at_lines(p.A, p.lda, p.sA) || !at_lines(p.B, p.ldb, p.sB)) split += work.tile_ktiles[kind];
  }
  return 4.0 * split > 3.0 * all;
}
TileKind small_tile_kind_of(const PlannedGemm* plans, const int* members, int n) {
  return has_wide_rows(plans, members, n) ? kTiles128 : small_tile_kind(work_of(plans, members, n));
}

int launch_tiles(PlannedGemm* plans, const int* members, int n, hipStream_t stream) {
  const TileKind kind = small_tile_kind_of(plans, members, n);
  TileLaunch launch;
  if (int rc = fill_launch(plans, members, n, kTileShapes[kind].m, kTileShapes[kind].n, &launch)) return rc;
  if (has_wide_rows(plans, members, n)) return launch_tiles_as<GemmTiles<2, 2, 4, 4, 2>, 2, true>(launch, stream);
  switch (kind) {
    case kTiles64: {
      // Tiles that leave a compute unit with one workgroup or two are requested further ahead: nothing else covers their
      // requests.  Two per unit hold three k-tiles each (A as late as B); more of them, short contractions, whose operands
      // stay in an XCD's 4 MB of L2, and rows that straddle cache lines, of which a unit can only have so many in flight,
      // lose by more than two (us, two / three / four k-tiles ahead, symmetric; tiles of a shorter contraction count by
      // their share of the longest):
      //   rows at cache lines     k 1024              1152                1408                3072                5376
      //   253 tiles          6.5 /  6.3 /  6.4    -                   -                  22.2 / 15.5 / 13.0  36.0 / 23.6 / 19.5
      //   300                7.6 /  7.9 /  8.2    8.3 /  8.5 / -     11.6 /  9.7 / -     22.6 / 19.0 / 19.9  36.4 / 30.8 / 32.2
      //   351                8.0 /  8.2 /  8.6    9.1 /  8.8 / -     12.6 / 11.1 / -     23.2 / 21.1 / 21.5  37.4 / 33.7 / 35.8
      //   406                8.5 /  8.7 /  8.9   10.1 /  9.5 / -     13.1 / 11.7 / -     23.5 / 22.0 / 22.0  38.4 / 34.6 / 36.9
      //   496                9.5 /  9.5 /  9.7   11.6 / 10.6 / -     13.6 / 12.5 / -     24.6 / 23.0 / 23.3  39.9 / 35.4 / 39.1
      //   528               11.0 / 12.1 / 13.6    -                   -                  24.6 / 30.1 / 30.8  40.1 / 48.8 / 51.1
      //   rows across them        k 1032              1160                1416                3080                5384
      //   253                7.4 /  7.3 /  7.4    -                   -                  23.2 / 18.8 / 18.7  37.1 / 29.4 / 29.5
      //   276                9.0 /  9.9 / -       9.5 / 10.6 / -     11.3 / 12.1 / -     23.5 / 23.1 / -     37.8 / 41.0 / -
      //   300                9.4 / 10.0 / 10.4   10.0 / 10.8 / -     12.5 / 12.5 / -     24.0 / 25.7 / 27.6  38.5 / 44.4 / 48.4
      //   406               11.3 / 11.5 / 11.6   12.7 / 13.2 / -     15.2 / 16.3 / -     27.5 / 32.0 / 32.3  47.5 / 53.6 / 53.5
      //   496               13.2 / 13.0 / 12.9   14.5 / 14.4 / -     17.1 / 17.2 / -     30.2 / 33.7 / 33.8  49.8 / 56.0 / 55.5
      const LaunchWork work = work_of(plans, members, n);
      const double long_tiles = work.tile_ktiles[kTiles64] / work.max_ktiles;
      if (long_tiles <= 256.0) return launch_tiles_as<GemmTiles<2, 2, 2, 2, 4>, 2>(launch, stream);
      if (long_tiles <= 500.0 && work.max_ktiles >= 18.0 && !has_split_rows(plans, members, n, kTiles64))
        return launch_tiles_as<GemmTiles<2, 2, 2, 2, 3, true>, 3>(launch, stream);
      return launch_tiles_as<GemmTiles<2, 2, 2, 2, 2>, 4>(launch, stream);
    }
    case kTiles128: {
      // Where some compute units have two of these tiles and others one, the ones with two are what a launch waits for.  If
      // rows straddle cache lines they have twice the lines to fetch, and the more of them in flight the slower (us with
      // A early / late; up to a round of two per unit):
      //   276 tiles, k 1032 22.8 / 21.0, k 3080 55.4 / 44.4   300, k 2056 41.8 / 33.2   384 with D, k 504 14.9 / 14.2
      // From there on all have as much to do, and the early requests are worth more (528, k 2056 63.8 / 70.8; with rows at
      // cache lines 276, k 2048 27.4 / 27.1 and 288 with D, k 1024 18.0 / 18.8).
      const LaunchWork work = work_of(plans, members, n);
      const double long_tiles = work.tile_ktiles[kTiles128] / work.max_ktiles;
      if (long_tiles > 256.0 && long_tiles <= kTileShapes[kTiles128].round && has_split_rows(plans, members, n, kTiles128))
        return launch_tiles_as<GemmTiles<2, 2, 4, 4, 2, true>, 2>(launch, stream);
      return launch_tiles_as<GemmTiles<2, 2, 4, 4, 2>, 2>(launch, stream);
    }
    case kTiles128Deep: return launch_tiles_as<GemmTiles<2, 2, 4, 4, 4>, 1>(launch, stream);
    // Eight waves: with four of 128 x 64 the start and the staged output of a tile took 2 to 3 us longer (us, four / eight:
    // 3400 x 3400 symmetric with D, k 3400 59.8 / 56.5   3200 x 3200 symmetric, k 3080 53.1 / 51.1
    // 8 x 2976 x 992, k 992, two outputs 72.8 / 65.5).
    default: return launch_tiles_as<GemmTiles<4, 2, 4, 4, 2>, 1>(launch, stream);
  }
}

// Launches the planned problems.  Problems that take the same kernel share
// launches: the short tiles of one problem then fill the partly empty last
// round of another instead of each launch paying its own start and tail.  The
// problems of one call must not depend on each other.
int launch_planned(PlannedGemm* plans, int count, hipStream_t stream) {
  for (int group = 0; group < 3; ++group) {  // large tiles, large tiles with k-major operands, small tiles
    const int limit = group < 2 ? GemmLaunch::kMaxProblems : TileLaunch::kMaxProblems;
    for (int next = 0; next < count;) {
      int members[TileLaunch::kMaxProblems];
      int n = 0;
      for (; next < count && n < limit; ++next)
        if (plans[next].large == (group < 2) && (group == 2 || plans[next].p.k_major == group)) members[n++] = next;
      if (n == 0) break;
      for (int a = 1; a < n; ++a)  // insertion sort, longest k first, stable
        for (int b = a; b > 0 && plans[members[b]].p.K > plans[members[b - 1]].p.K; --b) {
          const int t = members[b];
          members[b] = members[b - 1];
          members[b - 1] = t;
        }
      if (group == 2) {
        if (int rc = launch_tiles(plans, members, n, stream)) return rc;
      } else {
        GemmLaunch launch;
        if (int rc = fill_launch(plans, members, n, 256, 256, &launch)) return rc;
        if (int rc = launch_large_tiles(launch, group == 1, stream)) return rc;
      }
    }
  }
  return FSH_OK;
}

// Products of a Newton-Schulz iteration whose flow either kernel can serve:
// `plans[i].large` is set already where the flow asks for the large tiles; the
// others join them, all that fill a tile or none, if that is estimated to be
// faster by 10 %: two estimates are compared, each off by half of that.  One or
// two matrices of 2000 to 3300 a side come out so in their third product, whose
// tiles are a round and a bit on the small kernels and less than one here.
// Whole Muon steps, us: one 3072 x 3072 890 -> 798; 2248 x 2248 and 2176 x 2176
// 860 -> 782.  More than one round here is left alone: 20 matrices of 768 to
// 3072, whose last product is 1.4 rounds, were estimated 13 % faster for it and
// took 1 % longer (756 -> 764).
void choose_free_products(PlannedGemm* plans, int count) {
  LaunchWork in_large, rest, all;
  bool any = false;
  const auto candidate = [](const PlannedGemm& q) { return !q.large && q.fits && q.p.M >= 256 && q.p.N >= 256; };
  for (int i = 0; i < count; ++i) {
    const GemmParams& p = plans[i].p;
    if (plans[i].large) continue;
    const bool joins = candidate(plans[i]);
    any = any || joins;
    all.add(p.M, p.N, p.K, p.symmetric != 0, plans[i].batch);
    all.transposed = all.transposed || p.Ct != nullptr;
    LaunchWork& its = joins ? in_large : rest;
    its.add(p.M, p.N, p.K, p.symmetric != 0, plans[i].batch);
    its.transposed = its.transposed || p.Ct != nullptr;
  }
  if (!any || in_large.tiles[kTiles256] > kTileShapes[kTiles256].round) return;
  if (launch_us(kTiles256, in_large) + small_tiles_us(rest) >= 0.9 * small_tiles_us(all)) return;
  for (int i = 0; i < count; ++i) plans[i].large = plans[i].large || candidate(plans[i]);
}

// Plans `count` products that may share launches.  `large` (null: decided here):
// the problems that take the large-tile kernel at least.
constexpr int kPlannedTogether = 16;
int plan_gemms(const fsh_gemm_desc* descs, int count, const GemmUpdate* updates, const bool* large, PlannedGemm* plans) {
  for (int i = 0; i < count; ++i) {
    if (int rc = plan_gemm(descs[i], &plans[i], updates ? &updates[i] : nullptr)) return rc;
    if (large != nullptr) {
      plans[i].large = large[i];
      if (large[i] && !plans[i].fits) return fail(FSH_ENOTSUP, "gemm: a product does not fit the large tiles");
    }
  }
  if (large == nullptr) return choose_kernels(plans, count);
  choose_free_products(plans, count);
  return FSH_OK;
}
int launch_gemms(const fsh_gemm_desc* descs, int count, hipStream_t stream, const GemmUpdate* updates = nullptr,
                 const bool* large = nullptr) {
  PlannedGemm plans[kPlannedTogether];
  for (int begin = 0; begin < count; begin += kPlannedTogether) {
    const int n = count - begin < kPlannedTogether ? count - begin : kPlannedTogether;
    if (int rc = plan_gemms(descs + begin, n, updates ? updates + begin : nullptr, large ? large + begin : nullptr, plans)) return rc;
    if (int rc = launch_planned(plans, n, stream)) return rc;
  }
  return FSH_OK;
}

// The FSH_TILES_* that launch_planned takes for planned products.
void report_tiles(const PlannedGemm* plans, int count, int32_t* tiles) {
  for (int next = 0; next < count;) {  // the small-tile launches, as launch_planned fills them
    int members[TileLaunch::kMaxProblems], n = 0;
    for (; next < count && n < TileLaunch::kMaxProblems; ++next) {
      if (plans[next].large) tiles[next] = FSH_TILES_256;
      else members[n++] = next;
    }
    const TileKind kind = small_tile_kind_of(plans, members, n);
    for (int k = 0; k < n; ++k) tiles[members[k]] = kTileNames[kind];
  }
}

// A caller's k-major product: refused below 192 large tiles, where a
// transposed copy and the small tiles are faster.
int check_k_major(const fsh_gemm_desc& d) {
  if (!d.k_major || d.m <= 0 || d.n <= 0) return FSH_OK;
  if (count_tiles(d.m, d.n, d.symmetric != 0, 256, 256) * d.batch >= 192 && d.m % 256 == 0 && d.n % 256 == 0 && d.k % 64 == 0)
    return FSH_OK;
  return fail(FSH_ENOTSUP,
              "gemm: k-major operands need whole 256 x 256 x 64 tiles and at least 192 of them (m %lld, n %lld, "
              "k %lld, batch %lld)", (long long)d.m, (long long)d.n, (long long)d.k, (long long)d.batch);
}

float bf16_round_host(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
  memcpy(&f, &u, 4);
  return f;
}

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

}  // namespace
}  // namespace fsh

FSH_API int fsh_gemm_bf16_nt(const fsh_gemm_desc* desc, void* stream) {
  if (desc == nullptr) return fsh::fail(FSH_EINVAL, "fsh_gemm_bf16_nt: null descriptor");
  if (int rc = fsh::check_k_major(*desc)) return rc;
  return fsh::launch_gemms(desc, 1, static_cast<hipStream_t>(stream));
}

FSH_API int fsh_gemm_bf16_nt_group(const fsh_gemm_desc* descs, int32_t count, void* stream) {
  if (count < 0 || (count > 0 && descs == nullptr))
    return fsh::fail(FSH_EINVAL, "fsh_gemm_bf16_nt_group: bad descriptor list");
  for (int i = 0; i < count; ++i)
    if (int rc = fsh::check_k_major(descs[i])) return rc;
  return fsh::launch_gemms(descs, count, static_cast<hipStream_t>(stream));
}

FSH_API int fsh_gemm_bf16_tiles(const int64_t* sizes, int32_t count, int32_t* tiles) {
  using namespace fsh;
  if (count < 0 || count > kPlannedTogether || (count > 0 && (!sizes || !tiles))) return fail(FSH_EINVAL, "fsh_gemm_bf16_tiles: bad list");
  static __attribute__((aligned(16))) uint8_t somewhere[16];  // (looked at for its alignment alone)
  PlannedGemm plans[kPlannedTogether];
  for (int i = 0; i < count; ++i) {
    fsh_gemm_desc d;
    memset(&d, 0, sizeof(d));
    d.a_dev = d.b_dev = d.c_dev = somewhere;
    d.batch = sizes[5 * i]; d.m = sizes[5 * i + 1]; d.n = sizes[5 * i + 2]; d.k = sizes[5 * i + 3];
    d.symmetric = sizes[5 * i + 4] != 0;
    d.lda = d.ldb = d.k; d.ldc = d.n;
    d.stride_a = d.m * d.k; d.stride_b = d.n * d.k; d.stride_c = d.m * d.n;
    if (int rc = plan_gemm(d, &plans[i])) return rc;
  }
  if (int rc = choose_kernels(plans, count)) return rc;
  report_tiles(plans, count, tiles);
  return FSH_OK;
}

// Workspace layout (bytes, each region 256-aligned):
//   other orientation of the iterate [batch, s*l] bf16
//   second X^T buffer                [batch, s*l] bf16
//   G                                [batch, s*s] bf16
//   P                                [batch, s*s] bf16
//   norm partials                    [batch, slices_of(s*l / 8)] fp32
FSH_API int64_t fsh_newton_schulz_workspace_bytes(int64_t batch, int64_t rows, int64_t cols) {
  using namespace fsh;
  if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
  const int64_t s = rows < cols ? rows : cols, l = rows < cols ? cols : rows;
  return 2 * align256(batch * s * l * 2) + 2 * align256(batch * s * s * 2) +
         align256(batch * slices_of(ceil_div(s * l, (int64_t)8)) * 4);
}

namespace fsh {
namespace {

// One batch of equally shaped matrices on its way through the iteration.
// X is [s, l]; XT[0], XT[1] are the two [l, s] buffers.  The caller's buffer
// is X when the input is wide and XT[0] when it is tall.  The first X^T goes
// to XT[steps % 2] so that the last step leaves X^T in XT[0].
struct NsState {
  int64_t batch, s, l;
  uint16_t* X;
  uint16_t* XT[2];
  uint16_t* G;
  uint16_t* P;
  int cur;
  bool tall;    // the caller's matrix is X^T
  bool single;  // only X^T is carried from step to step (G = X X^T is then computed from its k-major rows)
};

// Workspace offset of the norm partials.
int64_t ns_partial_offset(int64_t batch, int64_t rows, int64_t cols) {
  const int64_t s = rows < cols ? rows : cols, l = rows < cols ? cols : rows;
  return 2 * align256(batch * s * l * 2) + 2 * align256(batch * s * s * 2);
}

// Which problems run on the large-tile kernel: all that consist of its whole
// tiles or none, whichever is estimated to take less time over an iteration's
// three products together with the other problems of the call (by a margin); then those with ragged edges
// as well, all whose short side fills a tile or none.  Whole Muon steps, us
// without / with ragged ones: one 5573 x 5573 and four small 4762 / 3434;
// 16 of 444 x 384, 1224 x 2176 and 1024 x 5248 4003 / 3176; 1 of 5494 x 4608
// and 16 of 256 x 5888 3232 / 2328; 16 of 832 x 2944, 334 x 960 and 2 of 2605 x
// 6784 3411 / 2712; 16 of 1100 x 1300 1182 / 941.
constexpr int64_t kRaggedLarge = 256;
double ns_iteration_us(const fsh_ns_problem* problems, int count, const bool* large) {
  double us = 0.0;
  for (int which = 0; which < 3; ++which) {
    LaunchWork in_large, small;
    for (int i = 0; i < count; ++i) {
      const fsh_ns_problem& q = problems[i];
      const int64_t s = q.rows < q.cols ? q.rows : q.cols, l = q.rows < q.cols ? q.cols : q.rows;
      const int64_t m = which == 2 ? l : s, k = which == 0 ? l : s;
      (large[i] ? in_large : small).add(m, s, k, which != 2, q.batch);
    }
    us += launch_us(kTiles256, in_large) + small_tiles_us(small);
  }
  return us;
}
void ns_choose_large(const fsh_ns_problem* problems, int count, int32_t steps, bool* large) {
  bool whole[FSH_MAX_NS_PROBLEMS], ragged[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    const fsh_ns_problem& q = problems[i];
    const int64_t s = q.rows < q.cols ? q.rows : q.cols, l = q.rows < q.cols ? q.cols : q.rows;
    large[i] = false;
    whole[i] = steps > 0 && s > 0 && s % 256 == 0 && l % 256 == 0 && l < (1LL << 22);
    ragged[i] = whole[i] || (steps > 0 && s >= kRaggedLarge && l < (1LL << 22));
  }
  double us = ns_iteration_us(problems, count, large);
  for (const bool* choice : {whole, ragged}) {
    const double with = ns_iteration_us(problems, count, choice);
    if (with >= kEstimateMargin * us) continue;
    us = with;
    for (int i = 0; i < count; ++i) large[i] = choice[i];
  }
}

// Checks a problem and lays out its buffers; `normalize` receives its part of
// the normalization launch.
int ns_begin(const fsh_ns_problem& q, bool large, int32_t steps, NsState* st, NormalizeGroup* normalize) {
  const int64_t batch = q.batch, rows = q.rows, cols = q.cols;
  if (batch <= 0 || rows <= 0 || cols <= 0)
    return fail(FSH_EINVAL, "newton_schulz: bad sizes (batch %lld, rows %lld, cols %lld)", (long long)batch,
                (long long)rows, (long long)cols);
  if (!q.x_dev || !q.workspace_dev) return fail(FSH_EINVAL, "newton_schulz: null pointer");
  if (rows % 8 || cols % 8)
    return fail(FSH_ENOTSUP, "newton_schulz: rows and cols must be multiples of 8, got %lld x %lld", (long long)rows,
                (long long)cols);
  if (!aligned(q.x_dev, 16) || !aligned(q.workspace_dev, 256))
    return fail(FSH_EINVAL, "newton_schulz: x must be 16-byte and workspace 256-byte aligned");
  if (batch > 65535) return fail(FSH_ENOTSUP, "newton_schulz: batch %lld exceeds 65535", (long long)batch);
  const int64_t need = fsh_newton_schulz_workspace_bytes(batch, rows, cols);
  if (q.workspace_nbytes < need)
    return fail(FSH_EINVAL, "newton_schulz: workspace of %lld bytes, need %lld", (long long)q.workspace_nbytes,
                (long long)need);
  const bool tall = rows > cols;
  const int64_t s = tall ? cols : rows, l = tall ? rows : cols;
  const int64_t sl = s * l, ss = s * s;
  uint8_t* ws = static_cast<uint8_t*>(q.workspace_dev);
  uint16_t* w0 = reinterpret_cast<uint16_t*>(ws);
  uint16_t* w1 = reinterpret_cast<uint16_t*>(ws + align256(batch * sl * 2));
  uint16_t* x = static_cast<uint16_t*>(q.x_dev);
  st->batch = batch;
  st->s = s;
  st->l = l;
  st->G = reinterpret_cast<uint16_t*>(ws + 2 * align256(batch * sl * 2));
  st->P = reinterpret_cast<uint16_t*>(ws + 2 * align256(batch * sl * 2) + align256(batch * ss * 2));
  float* partial = reinterpret_cast<float*>(ws + 2 * align256(batch * sl * 2) + 2 * align256(batch * ss * 2));
  // On the large-tile kernel G = X X^T is computed from X^T as it lies (k-major operands), so
  // X itself is never written: a tall input alternates between the caller's
  // buffer and one workspace buffer, a wide one between the two workspace
  // buffers and its last step writes X' = P X into the caller's buffer.
  st->single = large;
  st->X = tall ? w0 : x;
  st->XT[0] = tall ? x : w0;
  st->XT[1] = (st->single && tall) ? w0 : w1;
  st->cur = steps & 1;
  st->tall = tall;

  // Input is [rows, cols]; "same orientation" output is X for a wide input
  // and X^T for a tall one.
  uint16_t* same = tall ? st->XT[st->cur] : st->X;
  uint16_t* transposed = tall ? st->X : st->XT[st->cur];
  if (st->single) (tall ? transposed : same) = nullptr;
  normalize->in = x;
  normalize->out_same = same;
  normalize->out_t = transposed;
  normalize->partial = partial;
  normalize->rows = rows;
  normalize->cols = cols;
  const int64_t tiles_c = ceil_div(cols, (int64_t)kNormTile);
  const int64_t tiles = transposed ? tiles_c * ceil_div(rows, (int64_t)kNormTile) : ceil_div(rows * cols / 8, kSliceVectors);
  if (tiles >= INT32_MAX) return fail(FSH_ENOTSUP, "newton_schulz: more than %d blocks in one launch", INT32_MAX);
  normalize->tiles_c = static_cast<int32_t>(tiles_c);
  normalize->tiles = static_cast<int32_t>(tiles);
  normalize->slices = static_cast<int32_t>(slices_of(rows * cols / 8));
  return FSH_OK;
}

// Gives every group its block range: `blocks` per matrix of the group, `batch` matrices.
template <typename Group>
int add_blocks(Group* group, int64_t blocks, int64_t batch, int64_t* total) {
  group->first_block = static_cast<int32_t>(*total);
  *total += blocks * batch;
  if (*total >= INT32_MAX) return fail(FSH_ENOTSUP, "newton_schulz: more than %d blocks in one launch", INT32_MAX);
  return FSH_OK;
}

int launch_normalize(NormalizeLaunch& launch, const NsState* st, int count, float eps, hipStream_t stream) {
  int64_t blocks = 0, matrices = 0;
  for (int i = 0; i < count; ++i) {
    launch.group[i].first_matrix = static_cast<int32_t>(matrices);
    matrices += st[i].batch;  // (fewer than blocks)
    if (int rc = add_blocks(&launch.group[i], static_cast<int64_t>(launch.group[i].tiles), st[i].batch, &blocks)) return rc;
  }
  for (int i = count; i < kMaxMuonGroups; ++i) launch.group[i].first_block = launch.group[i].first_matrix = INT32_MAX;
  launch.eps_bf16 = bf16_round_host(eps);
  launch.norms_ready = 0;
  for (int i = 0; i < count; ++i) launch.norms_ready |= launch.group[i].slices > kNormSlices ? 1 : 0;
  if (launch.norms_ready) {
    hipLaunchKernelGGL(norm_groups_kernel, dim3(static_cast<uint32_t>(matrices)), dim3(kNormThreads), 0, stream, launch);
    if (int rc = check_launch("norm_groups_kernel")) return rc;
  }
  hipLaunchKernelGGL(normalize_groups_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, stream, launch);
  return check_launch("normalize_groups_kernel");
}

// One block per slice of every matrix of the groups for which `take` holds.
// Returns the number of blocks, or a negative error.
template <typename Take>
int64_t assign_slices(MuonLaunch& launch, const int64_t* batch, int count, Take take) {
  int64_t blocks = 0;
  // (groups left out get an empty range)
  for (int i = 0; i < count; ++i)
    if (int rc = add_blocks(&launch.group[i], take(i) ? launch.group[i].slices : 0, batch[i], &blocks)) return rc;
  for (int i = count; i < kMaxMuonGroups; ++i) launch.group[i].first_block = INT32_MAX;
  return blocks;
}

// The three products of one iteration; `which` = 0: G = X X^T, 1: P = a I +
// b G + c G G (symmetric because G is), 2: X' = P X = a X + (b G + c G G) X,
// also written transposed into the other X^T buffer -- or, when only X^T is
// carried, X'^T = X^T P alone, with G read from the k-major rows of X^T and
// the last step of a wide input written as X' = P X.  Carrying `a` on P's
// diagonal (added in fp32 before P is rounded) spares the last product a
// read of X from HBM per output tile.  The last step of the iteration writes
// only the orientation the caller holds: X' for a wide input, and for a tall
// one X'^T = X^T P (P is symmetric) computed directly.
fsh_gemm_desc ns_product(const NsState& st, int which, float a, float b, float c, bool last_step) {
  const int64_t s = st.s, l = st.l, sl = s * l, ss = s * s;
  fsh_gemm_desc g;
  memset(&g, 0, sizeof(g));
  g.batch = st.batch;
  if (which == 0 && st.single) {
    g.a_dev = st.XT[st.cur]; g.b_dev = st.XT[st.cur]; g.c_dev = st.G;
    g.m = s; g.n = s; g.k = l; g.lda = s; g.ldb = s; g.ldc = s;
    g.stride_a = sl; g.stride_b = sl; g.stride_c = ss;
    g.alpha = 1.0f; g.beta = 0.0f;
    g.symmetric = 1;
    g.k_major = 1;
  } else if (which == 0) {
    g.a_dev = st.X; g.b_dev = st.X; g.c_dev = st.G;
    g.m = s; g.n = s; g.k = l; g.lda = l; g.ldb = l; g.ldc = s;
    g.stride_a = sl; g.stride_b = sl; g.stride_c = ss;
    g.alpha = 1.0f; g.beta = 0.0f;
    g.symmetric = 1;
  } else if (which == 1) {
    g.a_dev = st.G; g.b_dev = st.G; g.d_dev = st.G; g.c_dev = st.P;
    g.m = s; g.n = s; g.k = s; g.lda = s; g.ldb = s; g.ldd = s; g.ldc = s;
    g.stride_a = ss; g.stride_b = ss; g.stride_d = ss; g.stride_c = ss;
    g.alpha = c; g.beta = b;
    g.diag_add = a;
    g.symmetric = 1;
  } else if (st.single ? (st.tall || !last_step) : (last_step && st.tall)) {
    // X'^T = X^T P (P is symmetric), the orientation that is carried
    g.a_dev = st.XT[st.cur]; g.b_dev = st.P; g.c_dev = st.XT[st.cur ^ 1];
    g.m = l; g.n = s; g.k = s; g.lda = s; g.ldb = s; g.ldc = s;
    g.stride_a = sl; g.stride_b = ss; g.stride_c = sl;
    g.alpha = 1.0f; g.beta = 0.0f;
  } else {
    g.a_dev = st.P; g.b_dev = st.XT[st.cur]; g.c_dev = st.X;
    g.ct_dev = (last_step || st.single) ? nullptr : st.XT[st.cur ^ 1];
    g.m = s; g.n = l; g.k = s; g.lda = s; g.ldb = s; g.ldc = l; g.ldct = s;
    g.stride_a = ss; g.stride_b = sl; g.stride_c = sl; g.stride_ct = sl;
    g.alpha = 1.0f; g.beta = 0.0f;
  }
  return g;
}

// The iteration proper for `count` normalized problems.
// `last_updates` (one per problem, or null): the last product of a problem
// whose entry has ptrs set applies that update to the parameters instead of
// writing the orthogonalized matrix to the caller's buffer.
int ns_iterate(NsState* st, int count, float a, float b, float c, int32_t steps, hipStream_t stream,
               const GemmUpdate* last_updates = nullptr) {
  fsh_gemm_desc descs[FSH_MAX_NS_PROBLEMS];
  bool large[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) large[i] = st[i].single;
  for (int step = 0; step < steps; ++step) {
    // The same product of every problem goes out together: problems are
    // independent of each other, the three products of one are not.
    for (int which = 0; which < 3; ++which) {
      const bool last = step + 1 == steps;
      for (int i = 0; i < count; ++i) descs[i] = ns_product(st[i], which, a, b, c, last);
      if (int rc = launch_gemms(descs, count, stream, last && which == 2 ? last_updates : nullptr, large)) return rc;
    }
    for (int i = 0; i < count; ++i) st[i].cur ^= 1;
  }
  // cur == 0 here: for a tall input the result X^T is in the caller's buffer;
  // for a wide input X was updated in place.
  return FSH_OK;
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_newton_schulz_tiles(const fsh_ns_problem* problems, int32_t count, int32_t steps, int32_t* large) {
  using namespace fsh;
  if (count < 0 || count > FSH_MAX_NS_PROBLEMS || (count > 0 && (!problems || !large)))
    return fail(FSH_EINVAL, "fsh_newton_schulz_tiles: bad list");
  bool takes_large[FSH_MAX_NS_PROBLEMS];
  ns_choose_large(problems, count, steps, takes_large);
  for (int i = 0; i < count; ++i) large[i] = takes_large[i] ? 1 : 0;
  return FSH_OK;
}

FSH_API int fsh_newton_schulz_product_tiles(const fsh_ns_problem* problems, int32_t count, int32_t steps, int32_t product,
                                            int32_t last_step, int32_t* tiles) {
  using namespace fsh;
  if (count < 0 || count > FSH_MAX_NS_PROBLEMS || (count > 0 && (!problems || !tiles)) || steps <= 0 || product < 0 || product > 2)
    return fail(FSH_EINVAL, "fsh_newton_schulz_product_tiles: bad list, step count or product");
  void* const somewhere = reinterpret_cast<void*>(static_cast<uintptr_t>(4096));  // (looked at for its alignment alone)
  bool large[FSH_MAX_NS_PROBLEMS];
  ns_choose_large(problems, count, steps, large);
  fsh_gemm_desc descs[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    fsh_ns_problem q = problems[i];
    q.x_dev = q.workspace_dev = somewhere;
    q.workspace_nbytes = fsh_newton_schulz_workspace_bytes(q.batch, q.rows, q.cols);
    NsState st;
    NormalizeGroup unused;
    if (int rc = ns_begin(q, large[i], steps, &st, &unused)) return rc;
    descs[i] = ns_product(st, product, 1.0f, 1.0f, 1.0f, last_step != 0);
  }
  PlannedGemm plans[kPlannedTogether];
  static_assert(FSH_MAX_NS_PROBLEMS <= kPlannedTogether, "one group of launches");
  if (int rc = plan_gemms(descs, count, nullptr, large, plans)) return rc;
  report_tiles(plans, count, tiles);
  return FSH_OK;
}

FSH_API int fsh_newton_schulz_multi(const fsh_ns_problem* problems, int32_t count, float a, float b, float c,
                                    int32_t steps, float eps, void* stream_) {
  using namespace fsh;
  if (count < 0 || count > FSH_MAX_NS_PROBLEMS || (count > 0 && problems == nullptr))
    return fail(FSH_EINVAL, "fsh_newton_schulz_multi: count %d outside [0, %d] or null list", count,
                FSH_MAX_NS_PROBLEMS);
  if (steps < 0) return fail(FSH_EINVAL, "fsh_newton_schulz_multi: negative step count %d", steps);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (count == 0) return FSH_OK;
  NsState st[FSH_MAX_NS_PROBLEMS];
  bool large[FSH_MAX_NS_PROBLEMS];
  ns_choose_large(problems, count, steps, large);
  NormalizeLaunch normalize;
  MuonLaunch sums;
  memset(&sums, 0, sizeof(sums));
  int64_t batch[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    if (int rc = ns_begin(problems[i], large[i], steps, &st[i], &normalize.group[i])) return rc;
    batch[i] = problems[i].batch;
    MuonGroupDev& g = sums.group[i];
    g.batch = static_cast<uint16_t*>(problems[i].x_dev);
    g.partial = normalize.group[i].partial;
    g.vectors = problems[i].rows * problems[i].cols / 8;
    g.slices = normalize.group[i].slices;
  }
  const int64_t blocks = assign_slices(sums, batch, count, [](int) { return true; });
  if (blocks < 0) return static_cast<int>(blocks);
  hipLaunchKernelGGL(sumsq_groups_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, stream, sums);
  if (int rc = check_launch("sumsq_groups_kernel")) return rc;
  if (int rc = launch_normalize(normalize, st, count, eps, stream)) return rc;
  return ns_iterate(st, count, a, b, c, steps, stream);
}

FSH_API int fsh_newton_schulz(void* x_dev, int64_t batch, int64_t rows, int64_t cols, float a, float b,
                              float c, int32_t steps, float eps, void* workspace_dev,
                              int64_t workspace_nbytes, void* stream_) {
  fsh_ns_problem q;
  q.x_dev = x_dev;
  q.batch = batch;
  q.rows = rows;
  q.cols = cols;
  q.workspace_dev = workspace_dev;
  q.workspace_nbytes = workspace_nbytes;
  return fsh_newton_schulz_multi(&q, 1, a, b, c, steps, eps, stream_);
}

// One Muon step over whole matrices grouped by shape: momentum (fused with
// the sum of squares), Newton-Schulz over all groups together, update.
FSH_API int fsh_muon_step(const fsh_muon_group* groups, int32_t count, float lerp_weight, float nesterov_weight,
                          int32_t nesterov, float decay_factor, float a, float b, float c, int32_t steps, float eps,
                          void* stream_) {
  using namespace fsh;
  if (count < 0 || count > FSH_MAX_NS_PROBLEMS || (count > 0 && groups == nullptr))
    return fail(FSH_EINVAL, "fsh_muon_step: count %d outside [0, %d] or null list", count, FSH_MAX_NS_PROBLEMS);
  if (steps < 0) return fail(FSH_EINVAL, "fsh_muon_step: negative step count %d", steps);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  fsh_ns_problem problems[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    const fsh_muon_group& g = groups[i];
    if (g.batch <= 0 || g.batch > 65535 || g.rows <= 0 || g.cols <= 0 ||
        ((g.rows % 8 || g.cols % 8) && g.layout != FSH_MUON_PADDED))
      return fail(FSH_EINVAL, "fsh_muon_step: group %d has bad sizes (batch %lld, rows %lld, cols %lld; rows and cols "
                  "must be multiples of 8 unless the layout is FSH_MUON_PADDED)", i, (long long)g.batch, (long long)g.rows,
                  (long long)g.cols);
    if (!g.param_ptrs_dev || !g.grad_ptrs_dev || !g.momentum_ptrs_dev || !g.batch_dev || !g.workspace_dev)
      return fail(FSH_EINVAL, "fsh_muon_step: group %d has a null pointer", i);
    if (!aligned(g.batch_dev, 16) || !aligned(g.workspace_dev, 256))
      return fail(FSH_EINVAL, "fsh_muon_step: group %d: batch buffer must be 16-byte and workspace 256-byte aligned", i);
    if (g.master_dtype != FSH_DT_BF16 && g.master_dtype != FSH_DT_F32)
      return fail(FSH_EINVAL, "fsh_muon_step: group %d: master_dtype %d is neither FSH_DT_BF16 nor FSH_DT_F32", i,
                  g.master_dtype);
    if (g.layout != 0 && g.layout != FSH_MUON_PADDED)
      return fail(FSH_EINVAL, "fsh_muon_step: group %d: unknown layout %d", i, g.layout);
    const int64_t rows = ceil_div(g.rows, (int64_t)8) * 8, cols = ceil_div(g.cols, (int64_t)8) * 8;
    if (g.workspace_nbytes < fsh_newton_schulz_workspace_bytes(g.batch, rows, cols))
      return fail(FSH_EINVAL, "fsh_muon_step: group %d: workspace of %lld bytes, need %lld", i,
                  (long long)g.workspace_nbytes, (long long)fsh_newton_schulz_workspace_bytes(g.batch, rows, cols));
    problems[i].x_dev = g.batch_dev;
    problems[i].batch = g.batch;
    problems[i].rows = rows;
    problems[i].cols = cols;
    problems[i].workspace_dev = g.workspace_dev;
    problems[i].workspace_nbytes = g.workspace_nbytes;
  }
  if (count == 0) return FSH_OK;
  NsState st[FSH_MAX_NS_PROBLEMS];
  bool large[FSH_MAX_NS_PROBLEMS];
  ns_choose_large(problems, count, steps, large);
  NormalizeLaunch normalize;
  MuonLaunch launch;
  memset(&launch, 0, sizeof(launch));
  launch.one_minus_mu = lerp_weight;
  launch.mu = nesterov_weight;
  launch.nesterov = nesterov;
  launch.decay = decay_factor;
  int64_t batch[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    if (int rc = ns_begin(problems[i], large[i], steps, &st[i], &normalize.group[i])) return rc;
    const fsh_muon_group& g = groups[i];
    batch[i] = g.batch;
    MuonGroupDev& q = launch.group[i];
    q.param_ptrs = g.param_ptrs_dev;
    q.momentum_ptrs = g.momentum_ptrs_dev;
    q.grad_ptrs = g.grad_ptrs_dev;
    q.batch = static_cast<uint16_t*>(g.batch_dev);
    q.partial = normalize.group[i].partial;
    q.vectors = problems[i].rows * problems[i].cols / 8;
    q.rows = g.rows;
    q.cols = g.cols;
    q.row_vectors = problems[i].cols / 8;
    q.slices = normalize.group[i].slices;
    q.f32 = g.master_dtype == FSH_DT_F32 ? 1 : 0;
    q.padded = g.rows % 8 || g.cols % 8 ? 1 : 0;
    q.neg_lr = g.neg_adjusted_lr;
    q.dir_scale = g.direction_scale;
  }
  int64_t blocks = assign_slices(launch, batch, count, [](int) { return true; });
  if (blocks < 0) return static_cast<int>(blocks);
  hipLaunchKernelGGL(muon_prepare_groups_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, stream, launch);
  if (int rc = check_launch("muon_prepare_groups_kernel")) return rc;
  if (int rc = launch_normalize(normalize, st, count, eps, stream)) return rc;
  // A group whose last product runs on the large-tile kernel gets its update
  // from that product's epilogue: the direction is never written and read
  // back.  The other groups' directions land in their batch buffers and a
  // separate launch applies them.
  GemmUpdate updates[FSH_MAX_NS_PROBLEMS];
  for (int i = 0; i < count; ++i) {
    // (the epilogue writes bf16 parameters in rows of 16-byte pieces; fp32 masters and odd widths take the separate launch)
    const bool fused = st[i].single && groups[i].master_dtype == FSH_DT_BF16 && !launch.group[i].padded;
    updates[i].ptrs = fused ? groups[i].param_ptrs_dev : nullptr;
    updates[i].decay = decay_factor;
    updates[i].neg_lr = groups[i].neg_adjusted_lr;
    updates[i].dir_scale = groups[i].direction_scale;
  }
  if (int rc = ns_iterate(st, count, a, b, c, steps, stream, updates)) return rc;
  blocks = assign_slices(launch, batch, count, [&](int i) { return updates[i].ptrs == nullptr; });
  if (blocks < 0) return static_cast<int>(blocks);
  if (blocks == 0) return FSH_OK;
  hipLaunchKernelGGL(muon_apply_groups_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, stream, launch);
  return check_launch("muon_apply_groups_kernel");
}

// ------------------------------------------------------------------------
// Allocation-free variant: the workspace is a static device array.
//
// `scratch` is a host-side stand-in for the device array, not a device
// address: each GPU holds its own copy at its own address, resolved once per
// device with hipGetSymbolAddress while that device is current.  Everything
// below uses the resolved pointer, never the array's name.
namespace fsh {
namespace {

// The norm partials of a batch that otherwise fills the scratch: 4 bytes for
// each slices_of() slice of a matrix, i.e. per 8192 elements or per matrix if it has
// fewer, and at most a quarter of the bytes are elements.
constexpr int64_t kScratchPartials = 1 << 20;
static __device__ __align__(256) uint8_t scratch[FSH_NS_STATIC_SCRATCH_BYTES + kScratchPartials];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// The current device's copy of `scratch`.
int static_scratch(void** out) {
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return fail(FSH_EHIP, "fsh_newton_schulz_noalloc: hipGetDevice: %s", hipGetErrorString(err));
  if (device < 0 || device >= kMaxDevices)
    return fail(FSH_ENOTSUP, "fsh_newton_schulz_noalloc: device index %d outside [0, %d)", device, kMaxDevices);
  void* ptr = g_scratch_ptr[device].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || ptr == nullptr)
      return fail(FSH_EHIP, "fsh_newton_schulz_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", device,
                  hipGetErrorString(err));
    g_scratch_ptr[device].store(ptr, std::memory_order_release);  // every thread resolves the same address
  }
  *out = ptr;
  return FSH_OK;
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_newton_schulz_noalloc(void* x_dev, int64_t batch, int64_t rows, int64_t cols, float a, float b,
                                      float c, int32_t steps, float eps, void* stream_) {
  using namespace fsh;
  if (batch <= 0 || rows <= 0 || cols <= 0)
    return fail(FSH_EINVAL, "fsh_newton_schulz_noalloc: bad sizes (batch %lld, rows %lld, cols %lld)", (long long)batch,
                (long long)rows, (long long)cols);
  // Checked in wide arithmetic before the byte count is formed: a huge request must not wrap around.
  const int64_t s = rows < cols ? rows : cols, l = rows < cols ? cols : rows;
  if (batch > 65535 || l > (1LL << 24) || s * l > FSH_NS_STATIC_SCRATCH_BYTES / 4 / batch)
    return fail(FSH_ENOTSUP,
                "fsh_newton_schulz_noalloc: batch %lld of %lld x %lld exceeds the %lld-byte static scratch; call "
                "fsh_newton_schulz with a workspace of fsh_newton_schulz_workspace_bytes()",
                (long long)batch, (long long)rows, (long long)cols, (long long)FSH_NS_STATIC_SCRATCH_BYTES);
  // The norm partials have room of their own behind the advertised size, against
  // which a matrix counts 64 of them, however many it has.
  const int64_t need = ns_partial_offset(batch, rows, cols) + align256(batch * 64 * 4);
  if (need > FSH_NS_STATIC_SCRATCH_BYTES || fsh_newton_schulz_workspace_bytes(batch, rows, cols) > FSH_NS_STATIC_SCRATCH_BYTES + kScratchPartials)
    return fail(FSH_ENOTSUP,
                "fsh_newton_schulz_noalloc: batch %lld of %lld x %lld needs %lld bytes of scratch, the static scratch "
                "holds %lld; call fsh_newton_schulz with a workspace of that size",
                (long long)batch, (long long)rows, (long long)cols, (long long)need,
                (long long)FSH_NS_STATIC_SCRATCH_BYTES);
  void* ptr = nullptr;
  if (int rc = static_scratch(&ptr)) return rc;
  // Every region of the workspace is written before it is read (norm
  // partials, both iterate buffers, G and P), so nothing has to be cleared
  // between calls.
  return fsh_newton_schulz(x_dev, batch, rows, cols, a, b, c, steps, eps, ptr,
                           FSH_NS_STATIC_SCRATCH_BYTES + kScratchPartials, stream_);
}

