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
// Matrix cores: v_mfma_f32_16x16x128_f8f6f4 (twice the rate of the 32x32x16 FP8
// form on gfx950).  A k-tile is one scale block (128 bytes of each row) and one
// such MFMA per block of 16 x 16: its partial product, from zero, is folded into
// the result with one fused multiply-add per element; the folds of one block run
// on the vector ALU while the matrix core works on the next ones.
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
// The half tile (128 x 256, waves of 32 x 128) is what the tiles of a last, at
// most half-full round are cut into.
using Fp8Gemm = Fp8Tile<4, 2, 4, 8, 2, 3>;
using Fp8GemmHalf = Fp8Tile<4, 2, 2, 8, 2, 6>;
static_assert(Fp8GemmHalf::kLdsBytes <= Fp8Gemm::kLdsBytes, "one launch holds both");

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
    fp8_gemm_tile<Fp8Gemm, kColumnScales>(p, lds_bytes, static_cast<int64_t>(uniform_i32(tm)) * Fp8Gemm::BM,
                                          static_cast<int64_t>(uniform_i32(tn)) * Fp8Gemm::BN);
  } else {
    // Same split over the XCDs as the whole tiles: the two halves of a tile are
    // neighbours in an XCD's run and share the tile's second operand in its L2.
    const int64_t id = static_cast<int64_t>(blockIdx.x) - p.whole_grid;
    const int64_t item = (id % kXcds) * p.half_items_per_xcd + id / kXcds;
    if (item >= p.half_items) return;
    tile_in_order(p.schedule, static_cast<int>(p.schedule.work_items + item / 2), &tm, &tn);
    const int64_t m0 = static_cast<int64_t>(uniform_i32(tm)) * Fp8Gemm::BM + uniform_i32(static_cast<int>(item & 1)) * Fp8GemmHalf::BM;
    if (m0 >= p.m) return;  // the second half of a tile that ends in its first (whole workgroup)
    fp8_gemm_tile<Fp8GemmHalf, kColumnScales>(p, lds_bytes, m0, static_cast<int64_t>(uniform_i32(tn)) * Fp8Gemm::BN);
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
// Measured (us with 64 x 64 tiles, 128 x 128, 256 x 256; block scales, the
// column-scale variant runs 5-10 % longer on all three; * fewer tiles than compute
// units, the deep form below), launches back to back on the same operands, and
// with the weight from memory:
//   48 x 14336, k 4096     11.1*  18.6*  24.2   15.4*  21.3*  32.9
//   1000 x 2048, k 5120    20.1   23.3*  31.6   25.0   27.6*  39.9
//   1000 x 5120, k 2048    19.9   16.9   15.5   24.4   21.5   18.5
//   553 x 12160, k 3456    42.7   29.9   35.2   49.0   33.8   43.9
//   3192 x 4736, k 1280    35.1   25.4   22.6   37.9   26.6   24.0
//   2295 x 3072, k 8960    97.2   66.2   60.5   105    76.2   65.2
//   144 x 3840, k 10240    22.0*  40.7*  55.8   512 x 4096, k 4096     15.3   19.0*  24.7  (the same operands only)
//   335 x 11136, k 10112   72.5   60.2   55.0   1400 x 4096, k 4096    39.1   30.2   27.7
//
// A compute unit with one workgroup to run has LDS to spare: more operand
// requests in flight ("deep").  Not where a unit runs several, whose requests
// cover one another's waits (us, fewer / more k-tiles in flight):
//   64 x 64:    48 x 14336, k 4096 12.9 / 10.8   144 x 3840, k 10240 26.9 / 22.0   1000 x 2048, k 5120 19.1 / 19.1
//               335 x 11136, k 10112 72.5 / 81.2   1000 x 5120, k 2048 20.2 / 21.5
//   128 x 128:  48 x 14336, k 4096 26.8 / 18.3   1000 x 2048, k 5120 32.5 / 23.1   1000 x 5120, k 2048 16.6 / 22.1
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
      {64, 64, 768.0, 0.20, 0.31, 0.58, 2.0},    // three workgroups per compute unit
      {128, 128, 512.0, 0.58, 0.66, 0.92, 4.0},  // two
      {128, 128, 256.0, 0.36, 0.40, 0.53, 4.0},  // one, deep
      {256, 256, 256.0, 0.50, 0.68, 1.46, 5.5},  // one; a round of at most half as many is cut into half tiles
  };
  const double ktiles = static_cast<double>(k / 128);
  int best = 0;
  double best_us = 0.0;
  int64_t best_tiles = 0;
  for (int i = 0; i < 4; ++i) {
    const int64_t tiles = ceil_div(m, kShapes[i].m) * ceil_div(n, kShapes[i].n);
    if ((i == 1 && tiles <= units) || (i == 2 && tiles > units)) continue;  // 128 x 128 is deep up to a tile per unit
    TileShape shape = kShapes[i];
    // A last round of more than half as many is not cut.  Us with 256 x 256 and 128 x 128 tiles, by the tiles of that round:
    //   132 33.5 / 29.7   144 35.2 / 29.9   135 22.3 / 18.8 (column scales, k 1408)
    //   143 38.3 / 48.3 (column scales, k 2944)   147 105 / 143   160 18.9 / 20.6   169 47.0 / 58.9   247 22.6 / 25.4
    if (i == 3 && units > 0 && 2 * (tiles % units) > units) shape.half = 1.2;
    const double us = rounds_us(shape, static_cast<double>(tiles), static_cast<double>(tiles) * ktiles, ktiles);
    if (i == 0 || us < best_us) {
      best = i;
      best_us = us;
      best_tiles = tiles;
    }
  }
  if (best == 0) return best_tiles <= (column_scales ? 2 * units : units) ? kFp8Tiles64Deep : kFp8Tiles64;
  if (best < 3) return best == 1 ? kFp8Tiles128 : kFp8Tiles128Deep;
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
  static LdsReservation reserved[2];
  const auto kernel = column_scales ? &fp8_gemm_tiles_kernel<Cfg, true, kBlocksPerUnit> : &fp8_gemm_tiles_kernel<Cfg, false, kBlocksPerUnit>;
  if (int rc = reserve_lds_once(reserved[column_scales], kernel, Cfg::kLdsBytes)) return rc;
  hipLaunchKernelGGL(kernel, grid, block, Cfg::kLdsBytes, stream, p);
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
  switch (fp8_tile_kind(p.m, p.n, p.k, column_scales, units)) {
    case kFp8Tiles64: return launch_fp8_tiles<Fp8Tile<2, 2, 2, 2, 3, 0>, 3>(p, column_scales, on);
    case kFp8Tiles64Deep: return launch_fp8_tiles<Fp8Tile<2, 2, 2, 2, 4, 2>, 2>(p, column_scales, on);
    case kFp8Tiles128: return launch_fp8_tiles<Fp8Tile<2, 2, 4, 4, 2, 3>, 2>(p, column_scales, on);
    case kFp8Tiles128Deep: return launch_fp8_tiles<Fp8Tile<2, 2, 4, 4, 4, 4>, 1>(p, column_scales, on);
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
